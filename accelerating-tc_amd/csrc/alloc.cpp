// Device memory of the contexts and the host side of transfers.
//
// hipMalloc and hipFree cost 20-300 us apiece at the sizes of a graph's
// buffers (hipFree also waits for the device): more than half of a one-shot
// count of a small or mid-sized graph.  A context keeps the blocks its buffers
// give back and gives them to its next buffers; a destroyed context leaves them
// to the device's other contexts, and the last one gives them back to the
// system.  A context keeps at most 1/16 of the device's memory, all of a device
// together 1/8: two contexts on graphs of R-MAT-23's size find their buffers again
// (with 1/16 for all of them a first count after another context's took 23.95
// instead of 23.0 ms).
// tc_ctx_release_memory gives it back, and so does every context when hipMalloc
// fails, which is then tried once more.
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <system_error>
#include <thread>

#include "internal.h"

namespace tcx {

struct Device;

struct Pool {
  std::mutex mu;
  std::multimap<size_t, void*> blocks;
  size_t held = 0;        // their bytes
  Device* dev = nullptr;  // null: nothing is kept
  bool closed = false;

  // Smallest kept block of at least `want` bytes that wastes little.
  void* take(size_t want, size_t* got);
  // Keeps the block, or returns false when it is not to be kept.
  bool give(void* p, size_t bytes);
  std::multimap<size_t, void*> drain();
};

namespace {

constexpr int kMaxDevices = 64;
constexpr int kCopyThreads = 4;
constexpr size_t kCopyChunk = 4u << 20;       // bytes per pinned slot, two slots a thread
constexpr size_t kStagedMin = 8u << 20;       // smaller copies go to the runtime as they are

// Pinned slots of one device's uploads (one upload at a time).
struct Staging {
  std::mutex mu;
  void* slot[2 * kCopyThreads] = {};
  hipEvent_t free_at[2 * kCopyThreads] = {};
};

}  // namespace

struct Device {
  // bytes kept by all pools, and how many may be by all and by each
  std::atomic<size_t> held{0}, cap{0}, cap_each{0};
  Pool shared;       // blocks of destroyed contexts: no work is pending on them
  int contexts = 0;
  Staging staging;
};

void* Pool::take(size_t want, size_t* got) {
  std::lock_guard<std::mutex> lk(mu);
  auto it = blocks.lower_bound(want);
  if (it == blocks.end() || it->first > (want < (1u << 20) ? 2 * want : want + want / 4))
    return nullptr;
  void* p = it->second;
  *got = it->first;
  held -= it->first;
  dev->held -= it->first;
  blocks.erase(it);
  return p;
}

bool Pool::give(void* p, size_t bytes) {
  if (!dev) return false;
  std::lock_guard<std::mutex> lk(mu);
  if (closed || held + bytes > dev->cap_each) return false;
  if (dev->held.fetch_add(bytes) + bytes <= dev->cap) {
    try {
      blocks.emplace(bytes, p);
      held += bytes;
      return true;
    } catch (const std::bad_alloc&) {  // a destructor may be giving it back
    }
  }
  dev->held -= bytes;
  return false;
}

std::multimap<size_t, void*> Pool::drain() {
  std::lock_guard<std::mutex> lk(mu);
  std::multimap<size_t, void*> out;
  out.swap(blocks);
  if (held) dev->held -= held;
  held = 0;
  return out;
}

namespace {

std::mutex g_mu;                              // registry
std::vector<std::weak_ptr<Pool>> g_pools;
Device g_dev[kMaxDevices];

thread_local Pool* t_pool = nullptr;
thread_local std::shared_ptr<Pool> t_owner;   // keeps t_pool alive

void free_blocks(std::multimap<size_t, void*> b) {
  for (auto& x : b) (void)hipFree(x.second);
}

void free_staging(Staging& s) {
  std::lock_guard<std::mutex> lk(s.mu);
  for (int i = 0; i < 2 * kCopyThreads; ++i) {
    if (s.free_at[i]) (void)hipEventDestroy(s.free_at[i]);
    if (s.slot[i]) (void)hipHostFree(s.slot[i]);
    s.free_at[i] = nullptr;
    s.slot[i] = nullptr;
  }
}

// Every kept block of every pool back to the system.
void trim_all() {
  std::lock_guard<std::mutex> lk(g_mu);
  for (auto& w : g_pools)
    if (auto p = w.lock()) free_blocks(p->drain());
  for (Device& d : g_dev) free_blocks(d.shared.drain());
}

// Sizes are rounded to an eighth of their power of two, so graphs of about
// the same size find each other's blocks.
size_t rounded(size_t want) {
  size_t g = 4096;
  while (16 * g <= want) g *= 2;
  return (want + g - 1) / g * g;
}

}  // namespace

PoolScope::PoolScope(const tc_ctx* c) : before(t_pool) {
  t_pool = c ? c->pool.get() : nullptr;
  if (c && c->pool) t_owner = c->pool;
}
PoolScope::~PoolScope() {
  t_pool = before;
  if (!t_pool) t_owner.reset();
}

std::shared_ptr<Pool> pool_create(int device, uint64_t total_mem) {
  std::shared_ptr<Pool> p;
  try {
    p = std::make_shared<Pool>();
    std::lock_guard<std::mutex> lk(g_mu);
    for (size_t i = 0; i < g_pools.size();)
      if (g_pools[i].expired()) g_pools.erase(g_pools.begin() + (long)i);
      else ++i;
    g_pools.push_back(p);
    if (device >= 0 && device < kMaxDevices) {
      Device& d = g_dev[device];
      d.contexts++;
      d.cap = (size_t)(total_mem / 8);
      d.cap_each = (size_t)(total_mem / 16);
      if (!d.shared.dev) d.shared.dev = &d;
      p->dev = &d;
    }
  } catch (const std::bad_alloc&) {
    return nullptr;
  }
  return p;
}

void pool_release(tc_ctx* c) {
  if (!c->pool || !c->pool->dev) return;
  free_blocks(c->pool->drain());
  free_blocks(c->pool->dev->shared.drain());
}

void pool_retire(std::shared_ptr<Pool> pool) {
  if (!pool || !pool->dev) return;
  {
    std::lock_guard<std::mutex> lk(pool->mu);
    pool->closed = true;
  }
  Device& d = *pool->dev;
  // under the registry's lock a new context neither uploads through the slots
  // nor finds blocks while the last one frees them
  std::lock_guard<std::mutex> lk(g_mu);
  std::multimap<size_t, void*> b = pool->drain();
  if (--d.contexts == 0) {
    free_blocks(std::move(b));
    free_blocks(d.shared.drain());
    free_staging(d.staging);
    return;
  }
  for (auto& x : b)
    if (!d.shared.give(x.second, x.first)) (void)hipFree(x.second);
}

int DevBuf::reserve(size_t want) {
  if (want <= bytes && p) return TC_OK;
  release();
  if (want == 0) want = 64;
  size_t size = want;
  if (t_pool && t_owner.get() == t_pool && t_owner->dev) {
    pool = t_owner;
    size = rounded(want);
    p = pool->take(size, &bytes);
    if (!p) p = pool->dev->shared.take(size, &bytes);
    if (p) return TC_OK;
  }
  hipError_t e = hipMalloc(&p, size);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    trim_all();
    e = hipMalloc(&p, size);
    if (e == hipErrorOutOfMemory && size > want) {  // without the rounding
      (void)hipGetLastError();
      size = want;
      e = hipMalloc(&p, size);
    }
  }
  if (e != hipSuccess) {
    p = nullptr;
    bytes = 0;
    pool.reset();
    (void)hipGetLastError();
    return fail(TC_ERR_NOMEM, "hipMalloc(%zu bytes) failed: %s", size, hipGetErrorString(e));
  }
  bytes = size;
  return TC_OK;
}

void DevBuf::release() {
  if (p && !(pool && pool->give(p, bytes))) (void)hipFree(p);
  p = nullptr;
  bytes = 0;
  pool.reset();
}

int fetch(tc_ctx* c, void* out, const void* src, size_t bytes) {
  if (bytes > kPinBytes) return fail(TC_ERR_RANGE, "fetch of %zu bytes", bytes);
  TCX_HIP(hipMemcpyAsync(c->pin, src, bytes, hipMemcpyDeviceToHost, c->stream));
  TCX_HIP(hipStreamSynchronize(c->stream));
  memcpy(out, c->pin, bytes);
  return TC_OK;
}

int fetch2(tc_ctx* c, uint64_t* out, const uint64_t* src, uint64_t* out2, const uint64_t* src2) {
  uint64_t* pin = static_cast<uint64_t*>(c->pin);
  TCX_HIP(hipMemcpyAsync(pin, src, 8, hipMemcpyDeviceToHost, c->stream));
  if (out2) TCX_HIP(hipMemcpyAsync(pin + 1, src2, 8, hipMemcpyDeviceToHost, c->stream));
  TCX_HIP(hipStreamSynchronize(c->stream));
  *out = pin[0];
  if (out2) *out2 = pin[1];
  return TC_OK;
}

// Pageable memory goes to the device at the speed of one host thread's copy
// into the runtime's pinned buffer (25 GB/s); four threads filling pinned
// slots of our own keep the link busy.
int upload(tc_ctx* c, void* dst, const void* src, size_t bytes) {
  if (bytes == 0) return TC_OK;
  Staging* s = c->device >= 0 && c->device < kMaxDevices ? &g_dev[c->device].staging : nullptr;
  std::unique_lock<std::mutex> lk;
  if (s && bytes >= kStagedMin) lk = std::unique_lock<std::mutex>(s->mu, std::try_to_lock);
  bool ready = lk.owns_lock();
  for (int i = 0; ready && i < 2 * kCopyThreads; ++i) {
    if (!s->slot[i] &&
        hipHostMalloc(&s->slot[i], kCopyChunk, hipHostMallocDefault) != hipSuccess) {
      s->slot[i] = nullptr;
      ready = false;
    }
    if (ready && !s->free_at[i] &&
        hipEventCreateWithFlags(&s->free_at[i], hipEventDisableTiming) != hipSuccess) {
      s->free_at[i] = nullptr;
      ready = false;
    }
  }
  if (!ready) {
    (void)hipGetLastError();
    TCX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c->stream));
    return TC_OK;
  }
  const size_t chunks = (bytes + kCopyChunk - 1) / kCopyChunk;
  hipError_t err[kCopyThreads] = {};
  auto work = [&](int t) {
    hipError_t e = hipSetDevice(c->device);
    for (size_t k = (size_t)t; e == hipSuccess && k < chunks; k += kCopyThreads) {
      const int i = 2 * t + (int)((k / kCopyThreads) & 1);
      const size_t at = k * kCopyChunk, len = std::min(kCopyChunk, bytes - at);
      e = hipEventSynchronize(s->free_at[i]);  // the slot's last copy is done
      if (e != hipSuccess) break;
      memcpy(s->slot[i], static_cast<const char*>(src) + at, len);
      e = hipMemcpyAsync(static_cast<char*>(dst) + at, s->slot[i], len, hipMemcpyHostToDevice,
                         c->stream);
      if (e == hipSuccess) e = hipEventRecord(s->free_at[i], c->stream);
    }
    err[t] = e;
  };
  std::thread th[kCopyThreads];
  int started = 1;
  try {
    for (; started < kCopyThreads; ++started) th[started] = std::thread(work, started);
  } catch (const std::system_error&) {
  }
  work(0);
  for (int t = started; t < kCopyThreads; ++t) work(t);  // threads that did not start
  for (int t = 1; t < started; ++t) th[t].join();
  for (hipError_t e : err)
    if (e != hipSuccess) return fail(TC_ERR_HIP, "staged upload failed: %s", hipGetErrorString(e));
  return TC_OK;
}

}  // namespace tcx

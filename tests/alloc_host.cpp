// The device memory of contexts (alloc.cpp) over a HIP runtime of this file: a
// card of kCard bytes whose blocks are host addresses.  Prints "ok", or what
// went wrong.
#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <random>
#include <thread>
#include <vector>

#include "../accelerating-tc_amd/csrc/internal.h"

constexpr size_t kCard = 1ull << 30;
static std::mutex g_card;
static std::map<void*, size_t> g_live;
static size_t g_used = 0, g_mallocs = 0;
static std::atomic<int> g_pinned{0}, g_events{0};
static std::atomic<long> g_copies_left{-1};  // copies until one fails (-1: none does)

static size_t used() {
  std::lock_guard<std::mutex> lk(g_card);
  return g_used;
}

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lk(g_card);
  ++g_mallocs;
  if (g_used + n > kCard) return hipErrorOutOfMemory;
  *p = malloc(16);
  g_live[*p] = n;
  g_used += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(g_card);
  auto it = g_live.find(p);
  if (it == g_live.end()) {
    printf("hipFree of a block that is not live\n");
    exit(1);
  }
  g_used -= it->second;
  g_live.erase(it);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return ++g_pinned, *p = malloc(n), hipSuccess; }
hipError_t hipHostFree(void* p) { return --g_pinned, free(p), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  return ++g_events, *e = reinterpret_cast<hipEvent_t>(8), hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return --g_events, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "out of memory"; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  if (g_copies_left >= 0 && g_copies_left-- == 0) return hipErrorUnknown;
  return memcpy(d, s, n), hipSuccess;
}
}

namespace tcx {
int fail(int status, const char*, ...) { return status; }
}  // namespace tcx

using tcx::DevBuf;

#define CHECK(x)                                        \
  do {                                                  \
    if (!(x)) {                                         \
      printf("line %d: %s\n", __LINE__, #x);            \
      exit(1);                                          \
    }                                                   \
  } while (0)

static tc_ctx* open_ctx() {
  tc_ctx* c = new tc_ctx();
  c->pool = tcx::pool_create(0, kCard);
  return c;
}
static void close_ctx(tc_ctx* c) {
  std::shared_ptr<tcx::Pool> p = c->pool;
  delete c;
  tcx::pool_retire(std::move(p));
}
// `count` buffers of `bytes` in use at once, then given back
static void use(tc_ctx* c, size_t bytes, int count) {
  tcx::PoolScope scope(c);
  std::vector<std::unique_ptr<DevBuf>> b;
  for (int i = 0; i < count; ++i) {
    b.emplace_back(new DevBuf());
    CHECK(b.back()->reserve(bytes) == TC_OK);
  }
}

int main() {
  // a context keeps 1/16 of the card, all of them together 1/8
  {
    tc_ctx* c = open_ctx();
    use(c, kCard / 64, 8);
    CHECK(used() > 0 && used() <= kCard / 16);
    close_ctx(c);
    CHECK(used() == 0);
  }
  std::vector<tc_ctx*> cs;
  for (int i = 0; i < 16; ++i) cs.push_back(open_ctx());
  for (tc_ctx* c : cs) use(c, kCard / 64, 4);
  CHECK(used() > 0 && used() <= kCard / 8);
  // a destroyed context's blocks count too
  for (int i = 8; i < 16; ++i) close_ctx(cs[i]);
  cs.resize(8);
  for (tc_ctx* c : cs) use(c, kCard / 64, 4);
  CHECK(used() > 0 && used() <= kCard / 8);

  // kept blocks are used again
  size_t before = g_mallocs;
  tcx::pool_release(cs[0]);
  for (tc_ctx* c : cs) tcx::pool_release(c);
  CHECK(used() == 0);
  use(cs[0], 1000000, 3);
  before = g_mallocs;
  for (int i = 0; i < 5; ++i) use(cs[0], 1000000, 3);
  CHECK(g_mallocs == before);

  // they are given back on request, and when an allocation fails
  tcx::pool_release(cs[0]);
  CHECK(used() == 0);
  for (tc_ctx* c : cs) use(c, kCard / 128, 1);
  CHECK(used() > 0);
  {
    tcx::PoolScope scope(cs[1]);
    DevBuf all;
    CHECK(all.reserve(kCard) == TC_OK);
    CHECK(used() == kCard);
    DevBuf more;
    CHECK(more.reserve(64) == TC_ERR_NOMEM && more.p == nullptr && more.bytes == 0);
  }
  // a request that fits, where its size rounded up does not
  {
    tcx::PoolScope scope(cs[1]);
    DevBuf most, rest;
    CHECK(most.reserve(kCard / 2) == TC_OK);
    CHECK(rest.reserve(kCard / 2 - 1000) == TC_OK);
  }
  // without a scope nothing is kept
  for (tc_ctx* c : cs) tcx::pool_release(c);
  {
    DevBuf b;
    CHECK(b.reserve(4096) == TC_OK);
  }
  CHECK(used() == 0);
  // a buffer that outlives its context
  {
    DevBuf b;
    tc_ctx* c = open_ctx();
    {
      tcx::PoolScope scope(c);
      CHECK(b.reserve(4096) == TC_OK);
    }
    close_ctx(c);
  }
  CHECK(used() == 0);
  for (tc_ctx* c : cs) close_ctx(c);
  CHECK(used() == 0);

  // a staged upload, any copy of which fails, says so, and the next one is whole
  {
    std::vector<char> src((9u << 20) + 5), dst(src.size());
    for (size_t i = 0; i < src.size(); ++i) src[i] = (char)(i * 7 + i / 4096);
    tc_ctx* c = open_ctx();
    for (long k = 0; k < 3; ++k) {
      g_copies_left = k;
      CHECK(tcx::upload(c, dst.data(), src.data(), src.size()) == TC_ERR_HIP);
      g_copies_left = -1;
      std::fill(dst.begin(), dst.end(), 0);
      CHECK(tcx::upload(c, dst.data(), src.data(), src.size()) == TC_OK && dst == src);
    }
    close_ctx(c);
  }

  // contexts that come and go on threads, with uploads through the shared slots
  std::vector<std::thread> th;
  for (int t = 0; t < 8; ++t)
    th.emplace_back([t] {
      std::mt19937_64 r(t);
      std::vector<char> src(9u << 20, (char)t), dst(9u << 20);
      for (int i = 0; i < 40; ++i) {
        tc_ctx* c = open_ctx();
        for (int j = 0; j < 5; ++j) use(c, 1 + r() % (kCard / 256), 1 + (int)(r() % 3));
        if (i % 8 == 0) {
          CHECK(tcx::upload(c, dst.data(), src.data(), src.size()) == TC_OK);
          CHECK(memcmp(dst.data(), src.data(), src.size()) == 0);
        }
        if (i % 3 == 0) tcx::pool_release(c);
        CHECK(used() <= kCard / 8 + 8 * 3 * (kCard / 256) * 9 / 8);
        close_ctx(c);
      }
    });
  for (auto& x : th) x.join();
  CHECK(used() == 0 && g_pinned == 0 && g_events == 0);
  printf("ok\n");
}

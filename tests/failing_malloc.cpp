// hipMalloc that counts its requests and fails on demand, loaded before the engine:
// the k-th request from fail_at(k) on is refused, with the retries that the engine
// makes of it.
#include <dlfcn.h>

#include <cstddef>

namespace {
long g_until = -1;      // requests before the refused one (-1: none is)
size_t g_size = 0;      // its first size
int g_refused = 0;      // attempts refused so far
long g_mallocs = 0;     // requests in all
constexpr int kOutOfMemory = 2;

size_t rounded(size_t want) {  // the engine's, so that a retry is told from a new request
  size_t g = 4096;
  while (16 * g <= want) g *= 2;
  return (want + g - 1) / g * g;
}
}  // namespace

extern "C" {
void fail_at(long k) {
  g_until = k;
  g_refused = 0;
}
// The refused request's size, 0 if none was made.
size_t failed() { return g_refused ? g_size : 0; }

long mallocs() { return g_mallocs; }

int hipMalloc(void** p, size_t n) {
  static auto real =
      reinterpret_cast<int (*)(void**, size_t)>(dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), "hipMalloc"));
  ++g_mallocs;
  if (g_until == 0) {
    if (!g_refused) g_size = n;
    // as asked, once more, and once without the rounding if there was any
    if (g_refused < 2 || (g_refused == 2 && n < g_size && rounded(n) == g_size)) {
      ++g_refused;
      return kOutOfMemory;
    }
    g_until = -1;
  } else if (g_until > 0) {
    --g_until;
  }
  return real(p, n);
}
}

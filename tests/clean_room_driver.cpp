// clean_room_driver.cpp -- hsdl_clean where device memory is short.  The driver's own
// hipMalloc and hipFree stand before the runtime's: they count what the library
// holds and can refuse a call.
//   clean_room_driver DUMP K room      the default form within what the least form takes
//   clean_room_driver DUMP K refused   every allocation of a clean refused in turn
#include <dlfcn.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "hsdl.h"

static std::mutex g_mu;
static std::map<void *, size_t> g_sizes;
static size_t g_held = 0, g_peak = 0, g_cap = ~(size_t)0;
static long g_calls = 0, g_refuse = -1;

extern "C" int hipMalloc(void **p, size_t n) {
  static auto real = (int (*)(void **, size_t))dlsym(RTLD_NEXT, "hipMalloc");
  std::lock_guard<std::mutex> g(g_mu);
  if (g_calls++ == g_refuse || g_held + n > g_cap) return 2;  // hipErrorOutOfMemory
  const int e = real(p, n);
  if (e) return e;
  g_sizes[*p] = n;
  g_held += n;
  if (g_held > g_peak) g_peak = g_held;
  return 0;
}
extern "C" int hipFree(void *p) {
  static auto real = (int (*)(void *))dlsym(RTLD_NEXT, "hipFree");
  std::lock_guard<std::mutex> g(g_mu);
  auto it = g_sizes.find(p);
  if (it != g_sizes.end()) {
    g_held -= it->second;
    g_sizes.erase(it);
  }
  return real(p);
}

struct Labels {
  std::vector<uint64_t> off;
  std::vector<uint32_t> hub;
  std::vector<uint8_t> hop;
  std::vector<int32_t> dist;
  bool operator==(const Labels &o) const {
    return off == o.off && hub == o.hub && hop == o.hop && dist == o.dist;
  }
};
static void must(int rc, const char *what) {
  if (rc == HSDL_OK) return;
  std::printf("%s: %d %s\n", what, rc, hsdl_last_error());
  std::exit(1);
}
static Labels labels(const hsdl_index *idx) {
  uint32_t n;
  uint8_t K;
  uint64_t total;
  must(hsdl_index_info(idx, &n, &K), "info");
  must(hsdl_label_count(idx, &total), "count");
  Labels l;
  l.off.resize(n + 1);
  l.hub.resize(total);
  l.hop.resize(total);
  l.dist.resize(total);
  must(hsdl_export_labels(idx, l.off.data(), l.hub.data(), l.hop.data(), l.dist.data()), "export");
  return l;
}
static hsdl_index *load(const char *path, int K) {
  hsdl_index *idx = nullptr;
  must(hsdl_load_labels(path, (uint8_t)K, 0, &idx), "load");
  must(hsdl_release_scratch(-1), "release");
  return idx;
}
static void form(const char *pairs, const char *copy) {
  setenv("HSDL_CLEAN_PAIRS", pairs, 1);
  setenv("HSDL_STREAM32", copy, 1);
}

int main(int argc, char **argv) {
  if (argc < 4) return 2;
  const int K = std::atoi(argv[2]);
  // the least form: tiles over the index's own labels
  form("0", "0");
  hsdl_index *idx = load(argv[1], K);
  const Labels before = labels(idx);
  const size_t base = g_held;
  g_peak = g_held;
  must(hsdl_clean(idx), "clean");
  const size_t least = g_peak - base;
  const Labels want = labels(idx);
  hsdl_free_index(idx);
  std::printf("least form: %zu bytes, %zu -> %zu labels\n", least, before.hub.size(),
              want.hub.size());
  std::fflush(stdout);
  if (want.hub.size() == before.hub.size()) return 1;

  if (!std::strcmp(argv[3], "room")) {
    for (const char *copy : {"1", "0"}) {
      form("1", copy);
      idx = load(argv[1], K);
      g_peak = g_held;
      g_cap = g_held + least;
      const int rc = hsdl_clean(idx);
      g_cap = ~(size_t)0;
      std::printf("default form, HSDL_STREAM32=%s, within it: %d\n", copy, rc);
      std::fflush(stdout);
      must(rc, "clean within the least form's memory");
      if (!(labels(idx) == want)) return 1;
      hsdl_free_index(idx);
    }
    std::puts("room done");
    return 0;
  }
  for (const char *pairs : {"0", "1", "2"}) {
    form(pairs, "1");
    int refused = 0, ok = 0;
    for (long at = 0;; ++at) {
      idx = load(argv[1], K);
      g_calls = 0;
      g_refuse = at;
      const int rc = hsdl_clean(idx);
      const bool met = g_calls > at;
      g_refuse = -1;
      if (rc == HSDL_ENOMEM) {
        ++refused;
        if (!(labels(idx) == before)) return 1;  // as it was, and the next clean works
        must(hsdl_clean(idx), "clean after a refused one");
      } else {
        must(rc, "clean");
        ++ok;
      }
      if (!(labels(idx) == want)) {
        std::printf("HSDL_CLEAN_PAIRS=%s, allocation %ld: wrong labels\n", pairs, at);
        return 1;
      }
      hsdl_free_index(idx);
      if (!met) break;
    }
    std::printf("HSDL_CLEAN_PAIRS=%s: %d refused, %d cleaned\n", pairs, refused, ok);
    std::fflush(stdout);
  }
  std::puts("refused done");
  return 0;
}

// Checks of the library's device memory bookkeeping (Arena, TmpArena,
// ScratchScope) on the CPU: the HIP allocation calls below stand in for a device
// of a given size.  Addresses are handed out but never touched.  The scenario is
// the first argument; the exit status is 0 when every check holds.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <random>
#include <vector>

#include "gp_dev.hpp"

namespace {
std::map<char *, size_t> g_live;          // allocations of the stand-in device
size_t g_held = 0, g_size = (size_t)1 << 40, g_peak = 0;
char *g_next = (char *)((uintptr_t)1 << 44);

#define CHECK(c)                                                  \
  do {                                                            \
    if (!(c)) {                                                   \
      std::printf("line %d: %s does not hold\n", __LINE__, #c); \
      std::exit(1);                                               \
    }                                                             \
  } while (0)
}  // namespace

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  if (n == 0 || g_held + n > g_size) { *p = nullptr; return hipErrorOutOfMemory; }
  *p = g_next;
  g_live[g_next] = n;
  g_next += (n + 4095) / 4096 * 4096;
  g_held += n;
  if (g_held > g_peak) g_peak = g_held;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  if (!p) return hipSuccess;
  auto it = g_live.find((char *)p);
  CHECK(it != g_live.end());              // freed twice, or never allocated
  g_held -= it->second;
  g_live.erase(it);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
}

using namespace gp;

namespace {

constexpr int64_t MB = (int64_t)1 << 20;

// a setup step that fails after its temporaries, some of them larger than the
// pool hands out
gp_status failing_step(bool small) {
  TmpArena tmp;
  char *a = nullptr, *b = nullptr, *c = nullptr;
  GP_TRY(tmp.alloc(&a, small ? MB : 600 * MB));
  GP_TRY(tmp.alloc(&b, 3 * MB));
  GP_TRY(tmp.alloc(&c, (int64_t)1 << 50));
  return GP_OK;
}

void failed_setup() {
  for (bool small : {true, false}) {
    {
      ScratchScope scope(nullptr);
      CHECK(failing_step(small) == GP_ERR_NOMEM);
    }
    CHECK(g_live.empty());
    CHECK(failing_step(small) == GP_ERR_NOMEM);   // without a scope
    CHECK(g_live.empty());
  }
}

// a long-lived buffer, and one larger than the pool hands out, on a device whose
// memory the pool's idle chunks hold
void idle_chunks() {
  g_size = (size_t)1200 * MB;
  {
    ScratchScope scope(nullptr);
    Arena keep;
    char *p = nullptr, *q = nullptr;
    for (int pass = 0; pass < 2; ++pass) {
      TmpArena tmp;
      char *t[8] = {};
      for (char *&x : t) CHECK(tmp.alloc(&x, 100 * MB) == GP_OK);
    }
    CHECK(g_held >= (size_t)800 * MB);   // idle, in the pool
    CHECK(keep.alloc(&p, 900 * MB) == GP_OK && p);
    TmpArena tmp;
    CHECK(tmp.alloc(&q, 250 * MB) == GP_OK && q);
    CHECK(keep.alloc(&p, 900 * MB) == GP_ERR_NOMEM && !p);
    keep.free_all();
    CHECK(tmp.alloc(&p, 700 * MB) == GP_OK && p);
    scratch_trim();                      // keeps the chunk of the buffer in use
    CHECK(g_held >= (size_t)950 * MB);
  }
  CHECK(g_live.empty());
}

// the byte counter of an arena is what it holds of the device, through random
// allocations and releases, on a large device and on one that refuses slabs
void bytes() {
  std::mt19937_64 rng(2);
  for (size_t size : {(size_t)1 << 40, (size_t)40 * MB}) {
    g_size = size;
    Arena a;
    std::vector<std::pair<char *, int64_t>> used;
    int64_t asked = 0;
    for (int step = 0; step < 4000; ++step) {
      if (used.empty() || rng() % 4) {
        const int64_t n = (int64_t)std::exp2((double)(rng() % 2500) / 100.0);
        char *p = nullptr;
        if (a.alloc(&p, n) != GP_OK) continue;
        used.push_back({p, n});
        asked += n;
      } else {
        const size_t i = rng() % used.size();
        char *p = used[i].first;
        a.release(p, used[i].second);
        CHECK(!p);
        asked -= used[i].second;
        used.erase(used.begin() + (long)i);
      }
      CHECK(a.bytes == (int64_t)g_held);
      CHECK(a.bytes >= asked);
    }
    a.free_all();
    CHECK(a.bytes == 0 && g_live.empty());
  }
}

// an arena that only counts comes to the bytes of one that allocates
void count_only() {
  std::mt19937_64 rng(3);
  for (int round = 0; round < 200; ++round) {
    Arena a, c;
    c.count_only = true;
    for (int i = 0; i < 60; ++i) {
      const int64_t n = rng() % 10 ? (int64_t)std::exp2((double)(rng() % 2500) / 100.0) : 0;
      char *p = nullptr, *q = (char *)&a;
      CHECK(a.alloc(&p, n) == GP_OK && c.alloc(&q, n) == GP_OK);
      CHECK(!q && a.bytes == c.bytes);
    }
    a.free_all();
    c.free_all();
    CHECK(g_live.empty());
  }
}

// random buffers of a scope: no two that are in use overlap, everything is given
// back, with idle chunks given back now and then and on a device too small for
// every request
void pool() {
  std::mt19937_64 rng(1);
  for (size_t size : {(size_t)1 << 40, (size_t)600 * MB}) {
    g_size = size;
    ScratchScope scope(nullptr);
    TmpArena tmp;
    std::map<char *, int64_t> used;
    int refused = 0;
    for (int step = 0; step < 20000; ++step) {
      if (rng() % 500 == 0) scratch_trim();
      if (used.empty() || rng() % 2) {
        const int64_t n = (int64_t)std::exp2((double)(rng() % 2900) / 100.0);
        char *p = nullptr;
        if (tmp.alloc(&p, n) != GP_OK) { ++refused; continue; }
        auto next = used.lower_bound(p);
        CHECK(next == used.end() || p + n <= next->first);
        if (next != used.begin()) { --next; CHECK(next->first + next->second <= p); }
        auto chunk = g_live.upper_bound(p);
        CHECK(chunk != g_live.begin());
        --chunk;
        CHECK(p + n <= chunk->first + chunk->second);
        used[p] = n;
      } else {
        auto it = used.begin();
        std::advance(it, (long)(rng() % used.size()));
        char *p = it->first;
        tmp.release(p, it->second);
        used.erase(it);
      }
    }
    CHECK(size > (size_t)1 << 38 ? refused == 0 : refused > 0);
    tmp.free_all();
    scratch_trim();
    CHECK(g_live.empty());
  }
}

}  // namespace

int main(int argc, char **argv) {
  const char *what = argc > 1 ? argv[1] : "";
  if (!std::strcmp(what, "failed_setup")) failed_setup();
  else if (!std::strcmp(what, "idle_chunks")) idle_chunks();
  else if (!std::strcmp(what, "pool")) pool();
  else if (!std::strcmp(what, "bytes")) bytes();
  else if (!std::strcmp(what, "count_only")) count_only();
  else { std::printf("unknown scenario '%s'\n", what); return 2; }
  return 0;
}

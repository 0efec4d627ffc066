// Checks of the library's device memory bookkeeping (Arena, TmpArena,
// ScratchScope) on the CPU: the HIP allocation calls below stand in for a device
// of a given size.  Addresses are handed out but never touched.  The scenario is
// the first argument; the exit status is 0 when every check holds.
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

}  // namespace

int main(int argc, char **argv) {
  const char *what = argc > 1 ? argv[1] : "";
  if (!std::strcmp(what, "failed_setup")) failed_setup();
  else { std::printf("unknown scenario '%s'\n", what); return 2; }
  return 0;
}

// gp_dev.hpp -- device-side internals shared by the HIP translation units:
// error macros, tracked device buffers and the gp_layout handle.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <iterator>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "gds2para.h"
#include "gp_grid.hpp"
#include "gp_status.hpp"

#define GP_HIP(call)                                                                    \
  do {                                                                                  \
    hipError_t _e = (call);                                                             \
    if (_e != hipSuccess)                                                               \
      return gp::fail(GP_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(_e)); \
  } while (0)

#define GP_TRY(call)                    \
  do {                                  \
    gp_status _s = (call);              \
    if (_s != GP_OK) return _s;         \
  } while (0)

namespace gp {

// Grid-stride launch helper: blocks of 256 threads, enough blocks to cover n.
inline unsigned blocks_for(int64_t n, int threads = 256) {
  int64_t b = (n + threads - 1) / threads;
  if (b < 1) b = 1;
  if (b > 2147483647LL) b = 2147483647LL;
  return (unsigned)b;
}

// Temporaries of one setup call (hierarchy, V0 basis, real AMG): those calls
// make thousands of short-lived buffers, and hipMalloc / hipFree (which waits
// for the device) took half of their time: 220 of 445 ms for the hierarchy at
// 128x128x16.  A ScratchScope keeps the memory of the temporary arenas
// (TmpArena) of its thread until it ends, carving buffers from a few chunks.
// A freed range is handed out again at once, which is safe because everything
// inside a scope runs on the scope's one stream; at its end the scope waits for
// that stream and gives everything back, so nothing outlives the call and no
// two threads share a pool.  Ranges that fit no request stay idle meanwhile: an
// allocation that fails gives the idle chunks back and tries again
// (device_malloc), and a caller that goes on to other large buffers inside its
// scope gives them back first (scratch_trim).
class ScratchPool {
 public:
  explicit ScratchPool(hipStream_t s) : s_(s) {}
  void *get(size_t bytes) {
    bytes = (bytes + 511) & ~(size_t)511;
    if (bytes > kDirect) return nullptr;
    auto best = free_.end();
    for (auto it = free_.begin(); it != free_.end(); ++it)
      if (it->second >= bytes && (best == free_.end() || it->second < best->second)) best = it;
    if (best == free_.end()) {
      size_t c = next_ > bytes ? next_ : bytes;
      void *p = nullptr;
      if (hipMalloc(&p, c) != hipSuccess) {
        (void)hipGetLastError();
        c = bytes;
        if (hipMalloc(&p, c) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
      }
      if (next_ < kChunkMax) next_ *= 2;
      chunk_[(char *)p] = c;
      best = free_.emplace((char *)p, c).first;
    }
    char *p = best->first;
    const size_t left = best->second - bytes;
    free_.erase(best);
    if (left) free_[p + bytes] = left;
    used_[p] = bytes;
    return p;
  }
  // false: not one of this pool's buffers
  bool put(void *q) {
    auto u = used_.find((char *)q);
    if (u == used_.end()) return false;
    char *p = u->first;
    size_t n = u->second;
    used_.erase(u);
    auto next = free_.lower_bound(p);
    if (next != free_.end() && next->first == p + n && !chunk_.count(next->first)) {
      n += next->second;
      next = free_.erase(next);
    }
    if (next != free_.begin() && !chunk_.count(p)) {
      auto prev = std::prev(next);
      if (prev->first + prev->second == p) { prev->second += n; return true; }
    }
    free_[p] = n;
    return true;
  }
  bool empty() const { return chunk_.empty(); }
  // Gives back the chunks that hold no buffer; false if there was none.
  bool trim() {
    bool any = false;
    for (auto c = chunk_.begin(); c != chunk_.end();) {
      auto f = free_.find(c->first);
      if (f == free_.end() || f->second != c->second) { ++c; continue; }
      if (!any) (void)hipStreamSynchronize(s_);
      any = true;
      (void)hipFree(c->first);
      free_.erase(f);
      c = chunk_.erase(c);
    }
    return any;
  }
  void drop() {
    for (auto &c : chunk_) (void)hipFree(c.first);
    chunk_.clear();
    free_.clear();
    used_.clear();
  }

 private:
  static constexpr size_t kDirect = (size_t)512 << 20;    // larger buffers are allocated by themselves
  static constexpr size_t kChunkMax = (size_t)256 << 20;
  hipStream_t s_;
  size_t next_ = (size_t)8 << 20;
  std::map<char *, size_t> chunk_, free_, used_;
};

inline thread_local ScratchPool *t_scratch = nullptr;

// hipMalloc; where it fails, once more after the thread's pool has given back
// its idle chunks.
inline hipError_t device_malloc(void **p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipSuccess) return e;
  (void)hipGetLastError();
  if (t_scratch && t_scratch->trim()) e = hipMalloc(p, bytes);
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

inline void scratch_trim() {
  if (t_scratch) (void)t_scratch->trim();
}

struct ScratchScope {
  explicit ScratchScope(hipStream_t s) : s_(s), outer_(t_scratch != nullptr), pool_(s) {
    if (!outer_) t_scratch = &pool_;
  }
  ~ScratchScope() {
    if (outer_) return;
    t_scratch = nullptr;
    if (pool_.empty()) return;
    (void)hipStreamSynchronize(s_);
    pool_.drop();
  }
  ScratchScope(const ScratchScope &) = delete;
  ScratchScope &operator=(const ScratchScope &) = delete;

 private:
  hipStream_t s_;
  bool outer_;
  ScratchPool pool_;
};

// Device allocation with a byte counter: what the arena holds of the device,
// slabs whole.  Buffers up to kSmall bytes are cut from slabs that live until
// free_all: a layout holds hundreds, and each hipMalloc / hipFree costs 40-200 us
// (38 of 134 ms of a whole 48x48x12 run was hipFree).  Slabs double from 64 KB to
// 32 MB, so their unused ends come to about as much again as the buffers in them
// at most; releasing a buffer cut from a slab frees nothing before free_all.
// With count_only set before the first call, nothing is allocated: alloc hands
// out null pointers and bytes becomes what the same calls would hold.
struct Arena {
  int64_t bytes = 0;
  bool count_only = false;
  template <class T>
  gp_status alloc(T **p, int64_t n) {
    *p = nullptr;
    if (n <= 0) return GP_OK;
    const size_t b = sizeof(T) * (size_t)n;
    void *q = nullptr;
    if (!tmp_ && b <= kSmall) {
      const size_t need = (b + 255) & ~(size_t)255;
      if (need > slab_left_) {
        const size_t size = slab_next_ > need ? slab_next_ : need;
        if (count_only || hipMalloc(&q, size) == hipSuccess) {
          keep(q, size, true);
          slab_ = (char *)q;
          slab_left_ = size;
          if (slab_next_ < ((size_t)32 << 20)) slab_next_ *= 2;
        } else {
          (void)hipGetLastError();
        }
        q = nullptr;
      }
      if (need <= slab_left_) {
        slab_left_ -= need;
        if (count_only) return GP_OK;
        *p = (T *)slab_;
        slab_ += need;
        return GP_OK;
      }
    }
    if (tmp_ && t_scratch) q = t_scratch->get(b);
    if (!q && !count_only && device_malloc(&q, b) != hipSuccess)
      return fail(GP_ERR_NOMEM, "hipMalloc of " + std::to_string(b) + " bytes failed");
    keep(q, b, false);
    *p = (T *)q;
    return GP_OK;
  }
  template <class T>
  void release(T *&p, int64_t) {
    if (!p) return;
    for (Held &h : held_)
      if (h.p == (void *)p) {
        // the first buffer of a slab shares the slab's address: it stays with the rest of it
        if (!h.slab) { give_back(h.p); bytes -= (int64_t)h.size; h = Held(); }
        break;
      }
    p = nullptr;
  }
  void free_all() {
    for (Held &h : held_)
      if (h.p) give_back(h.p);
    held_.clear();
    bytes = 0;
    slab_ = nullptr;
    slab_left_ = 0;
    slab_next_ = kSlabFirst;
  }

 protected:
  bool tmp_ = false;

 private:
  static constexpr size_t kSmall = (size_t)8 << 20, kSlabFirst = (size_t)64 << 10;
  struct Held {
    void *p = nullptr;
    size_t size = 0;
    bool slab = false;
  };
  std::vector<Held> held_;
  char *slab_ = nullptr;
  size_t slab_left_ = 0, slab_next_ = kSlabFirst;
  void keep(void *q, size_t size, bool slab) {
    bytes += (int64_t)size;
    if (count_only) return;
    Held h;
    h.p = q;
    h.size = size;
    h.slab = slab;
    held_.push_back(h);
  }
  void give_back(void *q) {
    if (!(tmp_ && t_scratch && t_scratch->put(q))) (void)hipFree(q);
  }
};

// Buffers that live for one function, whichever way it is left: from the
// thread's ScratchScope, if one is open (and then opened before the TmpArena),
// else allocated as they are.
struct TmpArena : Arena {
  TmpArena() { tmp_ = true; }
  ~TmpArena() { free_all(); }
  TmpArena(const TmpArena &) = delete;
  TmpArena &operator=(const TmpArena &) = delete;
};

// Deep host copy of a gp_mesh so the caller's arrays may be released.
struct HostMesh {
  gp_mesh view{};
  std::vector<double> xn, yn, zn, epsn, sign, side_area;
  std::vector<int32_t> mark_edge, mark_node, cdt_mark_port, port_side_ptr, side_dir, side_cnd;
  std::vector<int64_t> bd_edges, bd_nodes, side_edge_ptr, side_edges;
  void copy_from(const gp_mesh &m);
};

struct CsrD {            // FP64 CSR, int64 row pointers, int32 columns
  int64_t n = 0, nnz = 0;
  int64_t *rp = nullptr;
  int32_t *ci = nullptr;
  double *v = nullptr;
};

struct V0Data;           // defined in v0.hip
struct V0Path;           // defined in v0path.hip
void destroy_v0path(V0Path *);
// the column vectors that V0 solves keep: their bytes; giving them back (false:
// none were held)
int64_t v0path_work_bytes(const V0Path *);
bool trim_v0path(V0Path *);
int64_t v0path_bytes(const V0Path *);
struct Solver;           // defined in solver.hip
void destroy_v0(V0Data *);
void destroy_solver(Solver *);
int64_t solver_bytes(const Solver *);  // hierarchy, coarse cache and cached slot workspace
struct Hierarchy;
const Hierarchy *solver_hierarchy(const Solver *);

}  // namespace gp

namespace gp {
// Device time of one kernel class, measured with HIP events recorded on the
// launching stream around each launch, together with the algorithmic bytes of
// each launch (for the achieved-bandwidth figure).
struct KTimer {
  bool on = false;
  std::vector<hipEvent_t> ev;     // begin/end pairs
  std::vector<double> bytes;      // per pair
  size_t used = 0;
  void begin(hipStream_t s) {
    if (!on) return;
    if (2 * used + 2 > ev.size()) {
      for (int q = 0; q < 256; ++q) {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) { on = false; return; }
        ev.push_back(e);
      }
    }
    (void)hipEventRecord(ev[2 * used], s);
  }
  void end(hipStream_t s, double b) {
    if (!on) return;
    (void)hipEventRecord(ev[2 * used + 1], s);
    if (bytes.size() <= used) bytes.resize(used + 1);
    bytes[used] = b;
    ++used;
  }
  void reset() { used = 0; }
  ~KTimer() { for (hipEvent_t e : ev) (void)hipEventDestroy(e); }
};
}  // namespace gp

struct gp_layout {
  gp::KTimer ktimer;                    // level-0 edge smoother launches
  gp::HostMesh hm;
  gp::Grid g{};
  int64_t n = 0;                        // unknowns after PEC removal
  hipStream_t stream = nullptr;
  int32_t device = 0;                   // the device current when the layout was created
  gp::Arena arena;
  // device copy of the mesh contract
  double *xn = nullptr, *yn = nullptr, *zn = nullptr, *epsn = nullptr, *sign = nullptr;
  int32_t *mark_edge = nullptr, *mark_node = nullptr;
  uint8_t *rm_edge = nullptr, *bd_node = nullptr;
  int64_t *map_edge = nullptr, *map_edge_r = nullptr;
  // stiffness
  bool s_ready = false;
  gp::CsrD S;
  // V0 basis
  gp::V0Data *v0 = nullptr;
  // V0 quasi-static path: V0 operators in CSR and the Ad / Ac hierarchies,
  // built with the smoother v0_smoother names (gp_real_smoother)
  gp::V0Path *v0path = nullptr;
  int32_t v0_smoother = GP_SMOOTH_CHEBYSHEV;
  // solver hierarchy
  gp::Solver *solver = nullptr;
};

namespace gp {
gp_status ensure_device();
// exclusive scan of int64 counts (n entries) into offsets (n+1 entries) on the layout stream
gp_status exclusive_scan_i64(const int64_t *cnt, int64_t *off, int64_t n, hipStream_t s, Arena &tmp);
}  // namespace gp

// mg.hip -- multigrid hierarchy setup (GPU Galerkin products) and the
// split-form hybrid V-cycle, templated on the working precision.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <complex>
#include <type_traits>

#include <hipcub/hipcub.hpp>

#include "mg.hpp"

namespace gp {

namespace {

constexpr double kEps0v = kEps0;

// ---------------------------------------------------------------- setup kernels

// K0 = W * [S, eps_r eps0 on the diagonal, sigma on the diagonal]
__global__ void k_level0_K(int64_t n, const int64_t *__restrict__ rp, const int32_t *__restrict__ ci,
                           const double *__restrict__ s, const double *__restrict__ W, const double *__restrict__ epsr,
                           const double *__restrict__ sig, int32_t *__restrict__ oci, double *__restrict__ o0,
                           double *__restrict__ o1, double *__restrict__ o2) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double w = W[i];
  for (int64_t p = rp[i]; p < rp[i + 1]; ++p) {
    const bool d = ci[p] == (int32_t)i;
    oci[p] = ci[p];
    o0[p] = w * s[p];
    o1[p] = d ? w * epsr[i] * kEps0v : 0.;
    o2[p] = d ? w * sig[i] : 0.;
  }
}

// d[i] = M_ii (0 when row i stores no diagonal entry)
__global__ void k_diag(int64_t n, const int64_t *__restrict__ rp, const int32_t *__restrict__ ci,
                       const double *__restrict__ v, double *__restrict__ d) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double x = 0.;
  for (int64_t p = rp[i]; p < rp[i + 1]; ++p)
    if (ci[p] == i) x = v[p];
  d[i] = x;
}

// Off-diagonal copy of a one-valued CSR: cnt[i] = entries of row i off the
// diagonal; then the entries in their order, and d[i] = M_ii
__global__ void k_offdiag_count(int64_t n, const int64_t *__restrict__ rp, const int32_t *__restrict__ ci,
                                int64_t *__restrict__ cnt) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int64_t c = 0;
  for (int64_t p = rp[i]; p < rp[i + 1]; ++p) c += ci[p] != i;
  cnt[i] = c;
}
__global__ void k_offdiag_fill(int64_t n, const int64_t *__restrict__ rp, const int32_t *__restrict__ ci,
                               const double *__restrict__ v, const int64_t *__restrict__ rp2, int32_t *__restrict__ ci2,
                               double *__restrict__ v2) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int64_t q = rp2[i];
  for (int64_t p = rp[i]; p < rp[i + 1]; ++p)
    if (ci[p] != i) { ci2[q] = ci[p]; v2[q] = v[p]; ++q; }
}

// B0 = W * [eps_r eps0, sigma] * G   (row scaling of the gradient)
__global__ void k_level0_B(int64_t n, const int64_t *__restrict__ rp, const double *__restrict__ g,
                           const double *__restrict__ W, const double *__restrict__ epsr, const double *__restrict__ sig,
                           double *__restrict__ o0, double *__restrict__ o1) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double a = W[i] * epsr[i] * kEps0v, b = W[i] * sig[i];
  for (int64_t p = rp[i]; p < rp[i + 1]; ++p) { o0[p] = a * g[p]; o1[p] = b * g[p]; }
}

__global__ void k_diag_l1(int64_t nr, const int64_t *__restrict__ rp, const int32_t *__restrict__ ci, int nv,
                          const double *__restrict__ v0, const double *__restrict__ v1, const double *__restrict__ v2,
                          double *__restrict__ d0, double *__restrict__ d1, double *__restrict__ d2,
                          double *__restrict__ l0, double *__restrict__ l1, double *__restrict__ l2) {
  // one wavefront per row (the conductor aggregate rows of the auxiliary
  // operators hold up to ~1e5 entries)
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64;
  const int lane = threadIdx.x & 63;
  if (i >= nr) return;
  const double *v[3] = {v0, v1, v2};
  double d[3] = {0, 0, 0}, l[3] = {0, 0, 0};
  for (int64_t p = rp[i] + lane; p < rp[i + 1]; p += 64) {
    const bool diag = ci[p] == (int32_t)i;
    for (int k = 0; k < nv; ++k) {
      if (diag) d[k] += v[k][p];
      else l[k] += fabs(v[k][p]);
    }
  }
  for (int off = 32; off > 0; off >>= 1)
    for (int k = 0; k < 3; ++k) { d[k] += __shfl_down(d[k], off, 64); l[k] += __shfl_down(l[k], off, 64); }
  if (lane != 0) return;
  double *dd[3] = {d0, d1, d2}, *ll[3] = {l0, l1, l2};
  for (int k = 0; k < nv; ++k) { dd[k][i] = d[k]; ll[k][i] = l[k]; }
}

__global__ void k_d2f_arr(int64_t n, const double *__restrict__ a, float *__restrict__ b) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (float)a[i];
}

gp_status smoother_data(Arena &A, const Csr &M, double **d, double **l, hipStream_t s) {
  for (int k = 0; k < M.nv; ++k) {
    GP_TRY(A.alloc(&d[k], M.nr));
    GP_TRY(A.alloc(&l[k], M.nr));
  }
  k_diag_l1<<<blocks_for(M.nr * 64), 256, 0, s>>>(M.nr, M.rp, M.ci, M.nv, M.v[0], M.nv > 1 ? M.v[1] : nullptr,
                                              M.nv > 2 ? M.v[2] : nullptr, d[0], M.nv > 1 ? d[1] : nullptr,
                                              M.nv > 2 ? d[2] : nullptr, l[0], M.nv > 1 ? l[1] : nullptr,
                                              M.nv > 2 ? l[2] : nullptr);
  GP_HIP(hipStreamSynchronize(s));
  return GP_OK;
}

gp_status to_f32(Arena &A, const double *src, int64_t n, float **dst, hipStream_t s) {
  GP_TRY(A.alloc(dst, std::max<int64_t>(n, 1)));
  if (n) k_d2f_arr<<<blocks_for(n), 256, 0, s>>>(n, src, *dst);
  return GP_OK;
}

}  // namespace

gp_status aux_smoother_data(Arena &A, const Csr &M, double **d, double **l, hipStream_t s) {
  return smoother_data(A, M, d, l, s);
}

gp_status d2f_copy(const double *src, float *dst, int64_t n, hipStream_t s) {
  if (n) k_d2f_arr<<<blocks_for(n), 256, 0, s>>>(n, src, dst);
  GP_HIP(hipGetLastError());
  return GP_OK;
}

namespace {

gp_status dense_host(const Csr &M, int which, int64_t nr, int64_t nc, std::vector<double> *out, hipStream_t s) {
  HostCsr h;
  GP_TRY(csr_host_copy(M, &h, which, s));
  out->assign(nr * nc, 0.0);
  for (int64_t i = 0; i < nr; ++i)
    for (int64_t p = h.rp[i]; p < h.rp[i + 1]; ++p) (*out)[i * nc + h.ci[p]] += h.v[p];
  return GP_OK;
}

}  // namespace

// Level-0 slot order of the edge smoother: rows sorted by (16 x 16-cell xy
// tile, plane, ix, iy, direction).  The reference numbering puts a row's
// couplings 40k (x-edges of the plane), 80k (z-edges) and 161k (planes above
// and below) rows away at 200 x 200 x 24, farther than one XCD's L2 holds
// while it works through that many rows; in tile order the rows in flight on
// an XCD are one compact block of the mesh and share their neighbours' lines.
constexpr int kTile = 16;

__global__ void k_tile_keys(int64_t n, const int64_t *__restrict__ map_r, Grid g, uint64_t *__restrict__ key,
                            int32_t *__restrict__ idx) {
  int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  int dir; int64_t iz, ix, iy;
  g.decode(map_r[r], dir, iz, ix, iy);
  const uint64_t nty = (uint64_t)(g.Ny / kTile + 1);
  const uint64_t tile = (uint64_t)(ix / kTile) * nty + (uint64_t)(iy / kTile);
  key[r] = (((tile * (uint64_t)(g.Nz + 1) + (uint64_t)iz) * (uint64_t)(g.Nx + 1) + (uint64_t)ix) *
                (uint64_t)(g.Ny + 1) + (uint64_t)iy) * 3u + (uint64_t)dir;
  idx[r] = (int32_t)r;
}

gp_status level0_order(gp_layout *lay, Arena &A, int32_t **order, hipStream_t s) {
  const int64_t n = lay->n;
  *order = nullptr;
  TmpArena tmp;
  uint64_t *k1, *k2;
  int32_t *i1;
  GP_TRY(tmp.alloc(&k1, n)); GP_TRY(tmp.alloc(&k2, n)); GP_TRY(tmp.alloc(&i1, n));
  GP_TRY(A.alloc(order, n));
  k_tile_keys<<<blocks_for(n), 256, 0, s>>>(n, lay->map_edge_r, lay->g, k1, i1);
  size_t bytes = 0;
  GP_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, k1, k2, i1, *order, (int)n, 0, 64, s));
  uint8_t *buf;
  GP_TRY(tmp.alloc(&buf, (int64_t)bytes));
  GP_HIP(hipcub::DeviceRadixSort::SortPairs(buf, bytes, k1, k2, i1, *order, (int)n, 0, 64, s));
  GP_HIP(hipStreamSynchronize(s));
  tmp.free_all();
  return GP_OK;
}

// ---- plane march of the level-0 edge smoother: block numbering and codes ----
constexpr int kMarchHalf = kTile / 2;  // ix columns per block

__global__ void k_march_blk(int64_t n, const int32_t *__restrict__ ord, const int64_t *__restrict__ map_r, Grid g,
                            int32_t *__restrict__ blk) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  int dir; int64_t iz, ix, iy;
  g.decode(map_r[ord[p]], dir, iz, ix, iy);
  const int64_t nty = g.Ny / kTile + 1;
  const int64_t tile = (ix / kTile) * nty + iy / kTile;
  blk[p] = (int32_t)((tile * (g.Nz + 1) + iz) * 2 + (ix % kTile) / kMarchHalf);
}

// start[b] = first position of block b (n past the last): position p writes
// the starts of the blocks (blk[p - 1], blk[p]]; a decreasing block number
// (positions out of block order) sets *bad
__global__ void k_march_start(int64_t n, int64_t nb, const int32_t *__restrict__ blk, int32_t *__restrict__ start,
                              int32_t *__restrict__ bad) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p > n) return;
  const int64_t lo = p == 0 ? -1 : (int64_t)blk[p - 1];
  const int64_t hi = p == n ? nb : (int64_t)blk[p];
  if (hi < lo) { *bad = 1; return; }
  for (int64_t b = lo + 1; b <= hi; ++b) start[b] = (int32_t)p;
}

__global__ void k_march_inv(int64_t n, const int32_t *__restrict__ ord, int32_t *__restrict__ inv) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) inv[ord[p]] = (int32_t)p;
}

// Codes of the stored entries of position p's row (the SELL copy's slice
// p >> 6, lane p & 63); counts, over the rows, the stored entries (high 32
// bits of *outside) and those read from global memory (low 32 bits)
__global__ void k_march_code(int64_t n, int nplane, const int64_t *__restrict__ base, const int32_t *__restrict__ w,
                             const int32_t *__restrict__ ci, const int32_t *__restrict__ inv,
                             const int32_t *__restrict__ blk, const int32_t *__restrict__ start,
                             int32_t *__restrict__ code, unsigned long long *__restrict__ outside) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long out = 0;
  if (p < n) {
    const int64_t sl = p >> 6;
    const int lane = (int)(p & 63);
    const int32_t b = blk[p];
    const int32_t tb = b >> 1, z = tb % nplane;
    const int64_t b0 = base[sl];
    const int wd = w[sl];
    for (int t = 0; t < wd; ++t) {
      const int64_t e = b0 + (int64_t)t * 64 + lane;
      const int32_t c = ci[e], cp = inv[c], bc = blk[cp];
      const int32_t tc = bc >> 1, zc = tc % nplane;
      if (tc - zc == tb - z && (bc & 1) == (b & 1) && zc >= z - 1 && zc <= z + 1) {
        code[e] = ((zc - z + 1) << 16) | (cp - start[bc]);
      } else {
        code[e] = (int32_t)(0x80000000u | (uint32_t)c);
        ++out;
      }
    }
    out += (unsigned long long)wd << 32;
  }
  // one atomic per wavefront
  for (int m = 32; m >= 1; m >>= 1) out += __shfl_xor(out, m);
  if ((threadIdx.x & 63) == 0 && out) atomicAdd(outside, out);
}

int march_lds_setup();

gp_status build_edge_march(gp_layout *lay, Arena &A, Hierarchy *H, hipStream_t s) {
  EdgeMarch &M = H->march;
  if (M.tried || H->L.size() < 2) return GP_OK;
  M.tried = true;
  const Sell &K = H->L[0].Ks;
  const int64_t n = lay->n;
  const Grid &g = lay->g;
  if (!K.nr || K.nr != n || !K.rows || n >= ((int64_t)1 << 31)) return GP_OK;
  const int64_t nty = g.Ny / kTile + 1, ntx = g.Nx / kTile + 1;
  M.ntile = ntx * nty;
  M.nplane = (int32_t)(g.Nz + 1);
  M.nblk = M.ntile * M.nplane * 2;
  if (M.nblk >= ((int64_t)1 << 30)) return GP_OK;
  TmpArena tmp;
  int32_t *blk, *inv, *bad;
  unsigned long long *outside;
  GP_TRY(tmp.alloc(&blk, n)); GP_TRY(tmp.alloc(&inv, n)); GP_TRY(tmp.alloc(&bad, 1));
  GP_TRY(tmp.alloc(&outside, 1));
  GP_TRY(A.alloc(&M.start, M.nblk + 1));
  GP_TRY(A.alloc(&M.code, std::max<int64_t>(K.nent, 1)));
  GP_HIP(hipMemsetAsync(bad, 0, sizeof(int32_t), s));
  GP_HIP(hipMemsetAsync(outside, 0, sizeof(unsigned long long), s));
  GP_HIP(hipMemsetAsync(M.code, 0, sizeof(int32_t) * std::max<int64_t>(K.nent, 1), s));
  k_march_blk<<<blocks_for(n), 256, 0, s>>>(n, K.rows, lay->map_edge_r, g, blk);
  k_march_start<<<blocks_for(n + 1), 256, 0, s>>>(n, M.nblk, blk, M.start, bad);
  k_march_inv<<<blocks_for(n), 256, 0, s>>>(n, K.rows, inv);
  k_march_code<<<blocks_for(n), 256, 0, s>>>(n, M.nplane, K.base, K.w, K.ci, inv, blk, M.start, M.code, outside);
  int32_t bad_h = 0;
  unsigned long long out_h = 0;
  std::vector<int32_t> st((size_t)M.nblk + 1);
  GP_HIP(hipMemcpyAsync(&bad_h, bad, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  GP_HIP(hipMemcpyAsync(&out_h, outside, sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
  GP_HIP(hipMemcpyAsync(st.data(), M.start, sizeof(int32_t) * st.size(), hipMemcpyDeviceToHost, s));
  GP_HIP(hipStreamSynchronize(s));
  tmp.free_all();
  int32_t maxb = 0;
  for (int64_t b = 0; b < M.nblk; ++b) maxb = std::max(maxb, st[b + 1] - st[b]);
  if (bad_h || st[M.nblk] != n || maxb >= (1 << 16)) {  // not in block order: leave the march off
    M.code = nullptr;
    M.start = nullptr;
    return GP_OK;
  }
  M.maxb = maxb;
  M.lds_max = march_lds_setup();
  M.outside = (int64_t)(out_h & 0xffffffffull);
  M.entries = (int64_t)(out_h >> 32);
  return GP_OK;
}

// Level-0 free nodes in the same tile order (keys from the node's plane and
// (ix, iy)), for the nodal operators N, G^T and Pn of level 0.
gp_status level0_node_order(const LevelGrid &L, Arena &A, int32_t **order, hipStream_t s) {
  const Grid &g = L.g;
  const int64_t nn = L.nn();
  std::vector<uint64_t> key((size_t)nn);
  const uint64_t nty = (uint64_t)(g.Ny / kTile + 1);
  for (int64_t f = 0; f < nn; ++f) {
    const int64_t v = L.nrev[f], iz = v / g.Nns, r = v - iz * g.Nns, ix = r / (g.Ny + 1), iy = r - ix * (g.Ny + 1);
    const uint64_t tile = (uint64_t)(ix / kTile) * nty + (uint64_t)(iy / kTile);
    key[f] = ((tile * (uint64_t)(g.Nz + 1) + (uint64_t)iz) * (uint64_t)(g.Nx + 1) + (uint64_t)ix) * (uint64_t)(g.Ny + 1) +
             (uint64_t)iy;
  }
  std::vector<int32_t> ord((size_t)nn);
  for (int64_t f = 0; f < nn; ++f) ord[f] = (int32_t)f;
  std::stable_sort(ord.begin(), ord.end(), [&](int32_t a, int32_t b) { return key[a] < key[b]; });
  GP_TRY(A.alloc(order, nn));
  GP_HIP(hipMemcpyAsync(*order, ord.data(), sizeof(int32_t) * nn, hipMemcpyHostToDevice, s));
  GP_HIP(hipStreamSynchronize(s));
  return GP_OK;
}

// Connected components of the auxiliary coarsest level (union-find on the
// pattern of NL[0] | NL[1]): the positions of each block in ascending coarse
// index, blocks by ascending size.  Gauss-Jordan on the whole matrix with
// partial pivoting keeps every row inside its own block (off-block entries
// are exact zeros, and x - 0 * v = x), so inverting each block on its own
// with the columns in the same order gives the same bits in far less work.
gp_status aux_coarse_blocks(Arena &A, AuxAMG &X, hipStream_t s) {
  const int64_t n = X.nL;
  if (n <= 0) return GP_OK;
  std::vector<int32_t> par(n);
  for (int64_t i = 0; i < n; ++i) par[i] = (int32_t)i;
  auto find = [&](int32_t a) {
    while (par[a] != a) { par[a] = par[par[a]]; a = par[a]; }
    return a;
  };
  for (int64_t i = 0; i < n; ++i)
    for (int64_t j = i + 1; j < n; ++j)
      if (X.NL[0][i * n + j] != 0.0 || X.NL[1][i * n + j] != 0.0 || X.NL[0][j * n + i] != 0.0 ||
          X.NL[1][j * n + i] != 0.0) {
        const int32_t a = find((int32_t)i), b = find((int32_t)j);
        if (a != b) par[std::max(a, b)] = std::min(a, b);
      }
  std::vector<int32_t> root(n), size(n, 0);
  for (int64_t i = 0; i < n; ++i) { root[i] = find((int32_t)i); ++size[root[i]]; }
  std::vector<int32_t> order(n);
  for (int64_t i = 0; i < n; ++i) order[i] = (int32_t)i;
  // by block size, then by block (its smallest index), then ascending index
  std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) {
    if (size[root[a]] != size[root[b]]) return size[root[a]] < size[root[b]];
    if (root[a] != root[b]) return root[a] < root[b];
    return a < b;
  });
  X.perm_h = order;
  X.boff_h.assign(1, 0);
  std::vector<int32_t> rowblk(n);
  std::vector<int64_t> ioff, aoff;
  X.inv_len = X.aug_len = 0;
  X.max_blk = 0;
  X.small_h.clear();
  X.big_h.clear();
  for (int64_t p = 0; p < n;) {
    const int32_t r = root[order[p]], b = size[r];
    const int32_t blk = (int32_t)X.boff_h.size() - 1;
    for (int32_t q = 0; q < b; ++q) rowblk[p + q] = blk;
    ioff.push_back(X.inv_len);
    aoff.push_back(X.aug_len);
    X.inv_len += (int64_t)b * b;
    X.aug_len += 2 * (int64_t)b * b;
    (b <= kBlockGJMax ? X.small_h : X.big_h).push_back(blk);
    X.max_blk = std::max(X.max_blk, b);
    p += b;
    X.boff_h.push_back((int32_t)p);
  }
  X.nblk = (int32_t)X.boff_h.size() - 1;
  GP_TRY(A.alloc(&X.perm, n)); GP_TRY(A.alloc(&X.rowblk, n)); GP_TRY(A.alloc(&X.boff, X.nblk + 1));
  GP_TRY(A.alloc(&X.ioff, X.nblk)); GP_TRY(A.alloc(&X.aoff, X.nblk));
  GP_TRY(A.alloc(&X.small, std::max<int64_t>((int64_t)X.small_h.size(), 1)));
  GP_HIP(hipMemcpyAsync(X.perm, X.perm_h.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(X.rowblk, rowblk.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(X.boff, X.boff_h.data(), sizeof(int32_t) * (X.nblk + 1), hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(X.ioff, ioff.data(), sizeof(int64_t) * X.nblk, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(X.aoff, aoff.data(), sizeof(int64_t) * X.nblk, hipMemcpyHostToDevice, s));
  if (!X.small_h.empty())
    GP_HIP(hipMemcpyAsync(X.small, X.small_h.data(), sizeof(int32_t) * X.small_h.size(), hipMemcpyHostToDevice, s));
  GP_HIP(hipStreamSynchronize(s));  // the host vectors above go out of scope
  return GP_OK;
}

// FP32 copies of every operator the mixed-precision V-cycle reads, added to
// an existing FP64 hierarchy (so a layout solved in FP64 first and in mixed
// precision afterwards keeps one hierarchy instead of building a second).
gp_status hierarchy_add_f32(gp_layout *lay, Arena &A, Hierarchy *H, hipStream_t s) {
  if (H->has_f32) return GP_OK;
  const int64_t n = H->L[0].ne;
  GP_TRY(to_f32(A, H->W, n, &H->Wf, s));
  for (MgLevel &L : H->L) {
    GP_TRY(csr_to_float(A, L.K, &L.Kf, s));
    for (int q = 0; q < 2; ++q)
      if (L.K.dg[q]) GP_TRY(to_f32(A, L.K.dg[q], L.ne, &L.Kf.dg[q], s));
    if (L.K.sdg) GP_TRY(to_f32(A, L.K.sdg, L.ne, &L.Kf.sdg, s));
    if (L.Ks.nr) {
      GP_TRY(sell_to_float(A, L.Ks, &L.Ksf, s)); GP_TRY(sell_to_float(A, L.Bs, &L.Bsf, s));
      GP_TRY(sell_to_float(A, L.Ns, &L.Nsf, s)); GP_TRY(sell_to_float(A, L.GTs, &L.GTsf, s));
      GP_TRY(sell_to_float(A, L.Ps, &L.Psf, s)); GP_TRY(sell_to_float(A, L.PTs, &L.PTsf, s));
      GP_TRY(sell_to_float(A, L.Pns, &L.Pnsf, s));
    }
    GP_TRY(csr_to_float(A, L.B, &L.Bf, s));
    GP_TRY(csr_to_float(A, L.N, &L.Nf, s));
    GP_TRY(csr_to_float(A, L.G, &L.Gf, s));
    GP_TRY(csr_to_float(A, L.GT, &L.GTf, s));
    if (L.P.nr) {
      GP_TRY(csr_to_float(A, L.P, &L.Pf, s));
      GP_TRY(csr_to_float(A, L.PT, &L.PTf, s));
      GP_TRY(csr_to_float(A, L.Pn, &L.Pnf, s));
      GP_TRY(csr_to_float(A, L.PnT, &L.PnTf, s));
    }
    for (int k = 0; k < 3; ++k) {
      GP_TRY(to_f32(A, L.kd[k], L.ne, &L.kdf[k], s));
      GP_TRY(to_f32(A, L.kl[k], L.ne, &L.klf[k], s));
    }
    for (int k = 0; k < 2; ++k) {
      GP_TRY(to_f32(A, L.nd[k], L.nn, &L.ndf[k], s));
      GP_TRY(to_f32(A, L.nl[k], L.nn, &L.nlf[k], s));
    }
  }
  GP_TRY(aux_add_f32(A, H, s));
  GP_HIP(hipStreamSynchronize(s));
  H->has_f32 = true;
  return GP_OK;
}

gp_status build_hierarchy(gp_layout *lay, Arena &A, Hierarchy *H, bool want_f32, int max_levels) {
  auto t0 = std::chrono::steady_clock::now();
  if (!lay->s_ready) GP_TRY(gp_assemble_stiffness(lay));
  hipStream_t s = lay->stream;
  ScratchScope scratch(s);
  const gp_mesh &m = lay->hm.view;
  std::vector<LevelGrid> grids(1);
  level0_grid(m, &grids[0]);
  LevelGrid &g0 = grids[0];
  const int64_t n = g0.ne();
  if (n != lay->n) return fail(GP_ERR_STATE, "level-0 edge count differs from the layout");
  // level-0 per-edge data
  std::vector<double> W, epsr(n), sig(n);
  std::vector<int16_t> mcode(n);
  if (m.nz > 16000) return fail(GP_ERR_ARG, "more than 16000 z-planes");
  edge_dual_volume(g0, &W);
  for (int64_t k = 0; k < n; ++k) {
    int64_t e = g0.erev[k];
    int64_t L = e / g0.g.El;
    epsr[k] = m.stack_epsn[L];
    sig[k] = m.mark_edge[e] != 0 ? m.stack_sign[L] : 0.;
    mcode[k] = (int16_t)(L * 2 + (m.mark_edge[e] != 0 ? 1 : 0));
  }
  GP_TRY(A.alloc(&H->mcode, n)); GP_TRY(A.alloc(&H->tab_eps, m.nz)); GP_TRY(A.alloc(&H->tab_sig, m.nz));
  GP_HIP(hipMemcpyAsync(H->mcode, mcode.data(), sizeof(int16_t) * n, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(H->tab_eps, m.stack_epsn, sizeof(double) * m.nz, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(H->tab_sig, m.stack_sign, sizeof(double) * m.nz, hipMemcpyHostToDevice, s));
  GP_TRY(A.alloc(&H->W, n)); GP_TRY(A.alloc(&H->epsr, n)); GP_TRY(A.alloc(&H->sig, n));
  GP_HIP(hipMemcpyAsync(H->W, W.data(), sizeof(double) * n, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(H->epsr, epsr.data(), sizeof(double) * n, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(H->sig, sig.data(), sizeof(double) * n, hipMemcpyHostToDevice, s));
  H->L.clear();
  H->L.emplace_back();
  {
    MgLevel &L0 = H->L[0];
    L0.ne = n;
    L0.nn = g0.nn();
    const CsrD &S = lay->S;
    GP_TRY(csr_alloc(A, n, n, S.nnz, 3, &L0.K));
    GP_HIP(hipMemcpyAsync(L0.K.rp, S.rp, sizeof(int64_t) * (n + 1), hipMemcpyDeviceToDevice, s));
    k_level0_K<<<blocks_for(n), 256, 0, s>>>(n, S.rp, S.ci, S.v, H->W, H->epsr, H->sig, L0.K.ci, L0.K.v[0], L0.K.v[1],
                                             L0.K.v[2]);
    GP_TRY(A.alloc(&H->sdiag, n));
    k_diag<<<blocks_for(n), 256, 0, s>>>(n, S.rp, S.ci, S.v, H->sdiag);
    HostCsr hg;
    build_gradient(g0, &hg);
    GP_TRY(csr_upload(A, hg, &L0.G, s));
    GP_TRY(csr_alloc(A, n, L0.nn, L0.G.nnz, 2, &L0.B));
    GP_HIP(hipMemcpyAsync(L0.B.rp, L0.G.rp, sizeof(int64_t) * (n + 1), hipMemcpyDeviceToDevice, s));
    GP_HIP(hipMemcpyAsync(L0.B.ci, L0.G.ci, sizeof(int32_t) * L0.G.nnz, hipMemcpyDeviceToDevice, s));
    k_level0_B<<<blocks_for(n), 256, 0, s>>>(n, L0.G.rp, L0.G.v[0], H->W, H->epsr, H->sig, L0.B.v[0], L0.B.v[1]);
    GP_HIP(hipStreamSynchronize(s));
    GP_TRY(transpose(A, L0.G, &L0.GT, s));
    GP_TRY(spgemm(A, L0.GT, L0.B, &L0.N, s));
  }
  // coarser levels
  while ((int)H->L.size() < max_levels && grids.back().ne() > 400) {
    LevelGrid c;
    if (!coarsen_grid(grids.back(), &c)) break;
    if (c.ne() == 0 || c.nn() == 0) break;
    MgLevel &F = H->L.back();
    HostCsr hp, hpn, hg;
    build_edge_prolongation(grids.back(), c, &hp);
    build_node_prolongation(grids.back(), c, &hpn);
    build_gradient(c, &hg);
    GP_TRY(csr_upload(A, hp, &F.P, s));
    GP_TRY(csr_upload(A, hpn, &F.Pn, s));
    GP_TRY(transpose(A, F.P, &F.PT, s));
    GP_TRY(transpose(A, F.Pn, &F.PnT, s));
    MgLevel Cl;
    Cl.ne = c.ne();
    Cl.nn = c.nn();
    TmpArena tmp;
    Csr tmpc;
    GP_TRY(spgemm(tmp, F.K, F.P, &tmpc, s));
    GP_TRY(spgemm(A, F.PT, tmpc, &Cl.K, s));
    csr_release(tmp, tmpc);
    GP_TRY(spgemm(tmp, F.B, F.Pn, &tmpc, s));
    GP_TRY(spgemm(A, F.PT, tmpc, &Cl.B, s));
    csr_release(tmp, tmpc);
    GP_TRY(spgemm(tmp, F.N, F.Pn, &tmpc, s));
    GP_TRY(spgemm(A, F.PnT, tmpc, &Cl.N, s));
    csr_release(tmp, tmpc);
    GP_TRY(csr_upload(A, hg, &Cl.G, s));
    GP_TRY(transpose(A, Cl.G, &Cl.GT, s));
    grids.push_back(std::move(c));
    H->L.push_back(Cl);
  }
  // smoother data and FP32 copies
  for (MgLevel &L : H->L) {
    GP_TRY(smoother_data(A, L.K, L.kd, L.kl, s));
    GP_TRY(smoother_data(A, L.N, L.nd, L.nl, s));
  }
  if (H->L.size() > 1) {
    // level 0: K_eps and K_sig are diagonal; keep them as per-row arrays so the
    // smoother streams one value per entry (the coarse levels are built already)
    MgLevel &L0 = H->L[0];
    GP_TRY(A.alloc(&L0.K.dg[0], n)); GP_TRY(A.alloc(&L0.K.dg[1], n));
    k_diag<<<blocks_for(n), 256, 0, s>>>(n, L0.K.rp, L0.K.ci, L0.K.v[1], L0.K.dg[0]);
    k_diag<<<blocks_for(n), 256, 0, s>>>(n, L0.K.rp, L0.K.ci, L0.K.v[2], L0.K.dg[1]);
    GP_HIP(hipStreamSynchronize(s));
    A.release(L0.K.v[1], L0.K.nnz);
    A.release(L0.K.v[2], L0.K.nnz);
    L0.K.nv = 1;
    // and the stiffness diagonal too: the smoother loads row i of u for K_eps
    // and K_sig anyway, so K_S's diagonal entry would gather that row twice
    GP_TRY(A.alloc(&L0.K.sdg, n));
    k_diag<<<blocks_for(n), 256, 0, s>>>(n, L0.K.rp, L0.K.ci, L0.K.v[0], L0.K.sdg);
  }
  if (H->L.size() > 1) {
    GP_TRY(level0_order(lay, A, &H->ord_e, s));
    GP_TRY(level0_node_order(grids[0], A, &H->ord_n, s));
  }
  for (size_t l = 0; l + 1 < H->L.size(); ++l) {  // the coarsest level is solved densely
    MgLevel &L = H->L[l];
    const int32_t *oe = l == 0 ? H->ord_e : nullptr, *on = l == 0 ? H->ord_n : nullptr;
    if (l == 0 && L.K.sdg) {  // level 0: the SELL copy of K holds the off-diagonal entries
      TmpArena tmp;
      Csr K2 = L.K;
      K2.sdg = nullptr; K2.dg[0] = K2.dg[1] = nullptr;
      int64_t *cnt;
      GP_TRY(tmp.alloc(&cnt, L.K.nr)); GP_TRY(tmp.alloc(&K2.rp, L.K.nr + 1));
      k_offdiag_count<<<blocks_for(L.K.nr), 256, 0, s>>>(L.K.nr, L.K.rp, L.K.ci, cnt);
      GP_TRY(exclusive_scan_i64(cnt, K2.rp, L.K.nr, s, tmp));
      GP_HIP(hipMemcpyAsync(&K2.nnz, K2.rp + L.K.nr, sizeof(int64_t), hipMemcpyDeviceToHost, s));
      GP_HIP(hipStreamSynchronize(s));
      GP_TRY(tmp.alloc(&K2.ci, std::max<int64_t>(K2.nnz, 1))); GP_TRY(tmp.alloc(&K2.v[0], std::max<int64_t>(K2.nnz, 1)));
      k_offdiag_fill<<<blocks_for(L.K.nr), 256, 0, s>>>(L.K.nr, L.K.rp, L.K.ci, L.K.v[0], K2.rp, K2.ci, K2.v[0]);
      GP_TRY(sell_from_csr(A, K2, &L.Ks, s, "L.K off-diagonal", oe));
      GP_HIP(hipStreamSynchronize(s));
      tmp.free_all();
      L.K.nsdg = L.K.nnz - K2.nnz;
    } else {
      GP_TRY(sell_from_csr(A, L.K, &L.Ks, s, "L.K", oe));
    }
    GP_TRY(sell_from_csr(A, L.B, &L.Bs, s, "L.B", oe));
    GP_TRY(sell_from_csr(A, L.N, &L.Ns, s, "L.N", on));
    GP_TRY(sell_from_csr(A, L.GT, &L.GTs, s, "L.GT", on));
    GP_TRY(sell_from_csr(A, L.P, &L.Ps, s, "L.P", oe));
    GP_TRY(sell_from_csr(A, L.PT, &L.PTs, s, "L.PT"));
    GP_TRY(sell_from_csr(A, L.Pn, &L.Pns, s, "L.Pn", on));
  }
  // coarsest level to the host, dense
  const MgLevel &C = H->L.back();
  H->neL = C.ne;
  H->nnL = C.nn;
  for (int k = 0; k < 3; ++k) GP_TRY(dense_host(C.K, k, C.ne, C.ne, &H->KL[k], s));
  for (int k = 0; k < 2; ++k) GP_TRY(dense_host(C.B, k, C.ne, C.nn, &H->BL[k], s));
  for (int k = 0; k < 2; ++k) GP_TRY(dense_host(C.N, k, C.nn, C.nn, &H->NL[k], s));
  GP_TRY(dense_host(C.GT, 0, C.nn, C.ne, &H->GTL, s));
  GP_HIP(hipStreamSynchronize(s));
  GP_TRY(build_aux(lay, A, H));
  GP_TRY(aux_coarse_blocks(A, H->aux, s));
  if (want_f32) GP_TRY(hierarchy_add_f32(lay, A, H, s));
  {  // dense coarsest data on the device, for the per-frequency inverses
    auto up = [&](const std::vector<double> &h, double **d) -> gp_status {
      GP_TRY(A.alloc(d, std::max<int64_t>((int64_t)h.size(), 1)));
      if (!h.empty()) GP_HIP(hipMemcpyAsync(*d, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice, s));
      return GP_OK;
    };
    for (int k = 0; k < 3; ++k) GP_TRY(up(H->KL[k], &H->KLd[k]));
    for (int k = 0; k < 2; ++k) {
      GP_TRY(up(H->BL[k], &H->BLd[k]));
      GP_TRY(up(H->NL[k], &H->NLd[k]));
      GP_TRY(up(H->aux.NL[k], &H->aux.NLd[k]));
    }
    GP_TRY(up(H->GTL, &H->GTLd));
    GP_HIP(hipStreamSynchronize(s));
  }
  GP_TRY(aux_coarse_eigen(A, H->aux, s));
  {
    Csr Sv;
    Sv.nr = lay->S.n; Sv.nc = lay->S.n; Sv.nnz = lay->S.nnz; Sv.rp = lay->S.rp; Sv.ci = lay->S.ci; Sv.nv = 1; Sv.v[0] = lay->S.v;
    GP_TRY(spgemm_ex(A, Sv, H->L[0].G, &H->SG, s, 1));
    GP_TRY(spgemm_ex(A, Sv, H->aux.Gx, &H->SGx, s, 1));
    GP_TRY(sell_from_csr(A, Sv, &H->Ss, s, "S", H->ord_e));  // S rows are level 0's rows
    // and in the reference's row order for single-column products: there a
    // wavefront's 64 rows are 64 consecutive rows, so its row-indexed reads
    // and its 16-byte writes of y are whole lines.  Measured at 200x200x24,
    // FP64 A(w) x with one column: 113.6 us in tile order, 106-108 in strips
    // of 8 cells in x with (plane, ix, direction, iy) inside, 105-106 here.
    GP_TRY(sell_from_csr(A, Sv, &H->Ss1, s, "S1", nullptr));
  }
  H->setup_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return GP_OK;
}


// ---------------------------------------------------------------- coarsest levels per frequency

namespace {

// out[i] = A0[i] - w^2 A1[i] + i w A2[i]; A0 may be null (zero), n entries per matrix
__global__ void k_form_freq(int64_t n, double w, const double *__restrict__ A0, const double *__restrict__ A1,
                            const double *__restrict__ A2, C2<double> *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double a1 = -w * w;
  out[i] = {(A0 ? A0[i] : 0.0) + a1 * A1[i], w * A2[i]};
}

// out = N^-1 G^T (nn x ne; N^-1 complex, G^T real and mostly zero)
__global__ void k_coarse_ng(int64_t nn, int64_t ne, const C2<double> *__restrict__ ninv, const double *__restrict__ gt,
                            C2<double> *__restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nn * ne) return;
  const int64_t a = t / ne, i = t - a * ne;
  C2<double> v = {0., 0.};
  for (int64_t b = 0; b < nn; ++b) {
    const double g = gt[b * ne + i];
    const C2<double> m = ninv[a * nn + b];
    v.x += m.x * g;
    v.y += m.y * g;
  }
  out[t] = v;
}

// Augmented [A_b | I] of every block b of the auxiliary coarsest level at
// angular frequency w, A_b = -w^2 NL0 + i w NL1 restricted to the block's
// coarse indices (perm), row-major b x 2b at aoff[b].  One workgroup per block.
__global__ void __launch_bounds__(256) k_blk_form(const int32_t *__restrict__ perm, const int32_t *__restrict__ boff,
                                                  const int64_t *__restrict__ aoff, int64_t na, double w,
                                                  const double *__restrict__ N0, const double *__restrict__ N1,
                                                  C2<double> *__restrict__ aug) {
  const int blk = blockIdx.x;
  const int o = boff[blk], b = boff[blk + 1] - o;
  C2<double> *A = aug + aoff[blk];
  const double a1 = -w * w;
  for (int64_t t = threadIdx.x; t < 2 * (int64_t)b * b; t += blockDim.x) {
    const int r = (int)(t / (2 * b)), c = (int)(t - (int64_t)r * 2 * b);
    C2<double> v;
    if (c < b) {
      const int64_t q = (int64_t)perm[o + r] * na + perm[o + c];
      v = {0.0 + a1 * N0[q], w * N1[q]};
    } else {
      v = {c - b == r ? 1.0 : 0.0, 0.0};
    }
    A[t] = v;
  }
}

// The inverse halves of the augmented blocks in `list` into the packed
// inverse (block b row-major b x b at ioff[b]).  One workgroup per block.
__global__ void __launch_bounds__(256) k_blk_extract(const int32_t *__restrict__ list, const int32_t *__restrict__ boff,
                                                     const int64_t *__restrict__ aoff, const int64_t *__restrict__ ioff,
                                                     const C2<double> *__restrict__ aug, C2<double> *__restrict__ inv) {
  const int blk = list[blockIdx.x];
  const int b = boff[blk + 1] - boff[blk];
  const C2<double> *A = aug + aoff[blk];
  C2<double> *I = inv + ioff[blk];
  for (int64_t t = threadIdx.x; t < (int64_t)b * b; t += blockDim.x) {
    const int r = (int)(t / b), c = (int)(t - (int64_t)r * b);
    I[t] = A[(int64_t)r * 2 * b + b + c];
  }
}

// one block's augmented matrix <-> a dense [A | I] for dense_inverse_batched,
// which takes the n x n matrix and keeps the augmentation to itself
__global__ void k_blk_to_dense(int b, const C2<double> *__restrict__ aug, C2<double> *__restrict__ a) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)b * b) return;
  const int64_t r = t / b, c = t - r * b;
  a[t] = aug[r * 2 * b + c];
}

}  // namespace

int64_t coarse_entry_bytes(const Hierarchy &H) {
  const int64_t ne = H.neL, nn = H.nnL;
  return (int64_t)sizeof(C2<double>) * (ne * ne + 2 * ne * nn + (H.aux.eig ? 0 : H.aux.inv_len));
}

namespace {

// (Re)writes the device pointer table, growing it when the slots outgrew it.
gp_status coarse_table_write(const Hierarchy &H, CoarseCache &C, hipStream_t s) {
  const int need = (int)C.e.size();
  if (need > C.cap || !C.tab) {
    int cap = std::max(16, C.cap);
    while (cap < need) cap *= 2;
    // the previous table may still be read by queued kernels: wait for them
    GP_HIP(hipStreamSynchronize(s));
    if (C.tab) {
      GP_HIP(hipFree((void *)C.tab));
      C.bytes -= (int64_t)sizeof(double *) * 4 * C.cap;
      C.tab = nullptr;
    }
    const double **tab = nullptr;
    if (device_malloc((void **)&tab, sizeof(double *) * 4 * (size_t)cap) != hipSuccess) {
      C.cap = 0;
      return fail(GP_ERR_NOMEM, "coarse cache table allocation failed");
    }
    C.tab = tab;
    C.cap = cap;
    C.bytes += (int64_t)sizeof(double *) * 4 * cap;
  }
  const int64_t ne = H.neL, nn = H.nnL;
  std::vector<const double *> h(4 * (size_t)C.cap, nullptr);
  for (int q = 0; q < need; ++q) {
    if (!C.e[q].mem) continue;
    C2<double> *b = (C2<double> *)C.e[q].mem;
    h[q] = (const double *)b;
    h[C.cap + q] = (const double *)(b + ne * ne);
    h[2 * C.cap + q] = (const double *)(b + ne * ne + ne * nn);
    h[3 * C.cap + q] = (const double *)(b + ne * ne + 2 * ne * nn);
  }
  GP_HIP(hipMemcpyAsync((void *)C.tab, h.data(), sizeof(double *) * h.size(), hipMemcpyHostToDevice, s));
  GP_HIP(hipStreamSynchronize(s));  // h goes out of scope
  C.stale = false;
  return GP_OK;
}

// Frees unpinned entries, least recently used first, until one more entry of
// `add` bytes fits the bounds (or no unpinned entry is left).
gp_status coarse_make_room(CoarseCache &C, int64_t add, hipStream_t s) {
  for (;;) {
    int live = 0;
    int64_t b = 0;
    for (const CoarseEntry &x : C.e)
      if (x.mem) { ++live; b += x.bytes; }
    if (live + 1 <= C.max_entries && b + add <= C.max_bytes) return GP_OK;
    int victim = -1;
    for (int q = 0; q < (int)C.e.size(); ++q)
      if (C.e[q].mem && C.e[q].pins == 0 && (victim < 0 || C.e[q].used < C.e[victim].used)) victim = q;
    if (victim < 0) return GP_OK;   // everything pinned: exceed the bound
    GP_HIP(hipStreamSynchronize(s));
    GP_HIP(hipFree(C.e[victim].mem));
    C.bytes -= C.e[victim].bytes;
    C.e[victim] = CoarseEntry{};
    ++C.evictions;
  }
}

}  // namespace

// The auxiliary coarsest level's inverse at angular frequency w, block by
// block (AuxAMG::nblk), packed into inv (block b at offset ioff[b]).
gp_status aux_coarse_inverse(const AuxAMG &X, double w, C2<double> *inv, hipStream_t s) {
  TmpArena T;
  struct Free { Arena &a; ~Free() { a.free_all(); } } fr{T};
  C2<double> *aug = nullptr;
  int *bad = nullptr;
  GP_TRY(T.alloc(&aug, std::max<int64_t>(X.aug_len, 1)));
  GP_TRY(T.alloc(&bad, 1));
  GP_HIP(hipMemsetAsync(bad, 0, sizeof(int), s));
  k_blk_form<<<X.nblk, 256, 0, s>>>(X.perm, X.boff, X.aoff, X.nL, w, X.NLd[0], X.NLd[1], aug);
  const unsigned nsmall = (unsigned)X.small_h.size();
  if (nsmall) {
    GP_TRY(gj_workgroup(X.small, X.boff, X.aoff, (int)nsmall, aug, bad, s));
    k_blk_extract<<<nsmall, 256, 0, s>>>(X.small, X.boff, X.aoff, X.ioff, aug, inv);
  }
  for (int32_t blk : X.big_h) {
    const int b = X.boff_h[blk + 1] - X.boff_h[blk];
    int64_t ao = 0, io = 0;
    for (int32_t q = 0; q < blk; ++q) {
      const int64_t bq = X.boff_h[q + 1] - X.boff_h[q];
      ao += 2 * bq * bq;
      io += bq * bq;
    }
    C2<double> *dst = inv + io;
    k_blk_to_dense<<<blocks_for((int64_t)b * b), 256, 0, s>>>(b, aug + ao, dst);
    GP_TRY(dense_inverse_batched(dst, b, 1, s));
  }
  int hbad = 0;
  GP_HIP(hipMemcpyAsync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost, s));
  GP_HIP(hipStreamSynchronize(s));
  if (hbad) return fail(GP_ERR_STATE, "singular block in the auxiliary coarsest level");
  return GP_OK;
}

gp_status aux_coarse_dense(const Hierarchy &H, double w, std::vector<std::complex<double>> *mat,
                           std::vector<std::complex<double>> *inv, hipStream_t s) {
  const AuxAMG &X = H.aux;
  const int64_t n = X.nL;
  mat->assign(n * n, 0.0);
  inv->assign(n * n, 0.0);
  if (n == 0) return GP_OK;
  for (int64_t q = 0; q < n * n; ++q) (*mat)[q] = {0.0 + (-w * w) * X.NL[0][q], w * X.NL[1][q]};
  if (X.eig) {
    std::vector<double> V(n * n), lam(n);
    GP_HIP(hipMemcpyAsync(V.data(), X.V, sizeof(double) * n * n, hipMemcpyDeviceToHost, s));
    GP_HIP(hipMemcpyAsync(lam.data(), X.lam, sizeof(double) * n, hipMemcpyDeviceToHost, s));
    GP_HIP(hipStreamSynchronize(s));
    std::vector<std::complex<double>> d(n);
    for (int64_t m = 0; m < n; ++m) d[m] = 1.0 / std::complex<double>(-w * w, w * lam[m]);
    for (int64_t i = 0; i < n; ++i)
      for (int64_t j = 0; j < n; ++j) {
        std::complex<double> acc = 0;
        for (int64_t m = 0; m < n; ++m) acc += V[i * n + m] * d[m] * V[j * n + m];
        (*inv)[i * n + j] = acc;
      }
    return GP_OK;
  }
  TmpArena T;
  struct Free { Arena &a; ~Free() { a.free_all(); } } fr{T};
  C2<double> *d = nullptr;
  GP_TRY(T.alloc(&d, std::max<int64_t>(X.inv_len, 1)));
  GP_TRY(aux_coarse_inverse(X, w, d, s));
  std::vector<std::complex<double>> h(X.inv_len);
  GP_HIP(hipMemcpyAsync(h.data(), d, sizeof(C2<double>) * X.inv_len, hipMemcpyDeviceToHost, s));
  GP_HIP(hipStreamSynchronize(s));
  int64_t io = 0;
  for (int32_t B = 0; B < X.nblk; ++B) {
    const int o = X.boff_h[B], b = X.boff_h[B + 1] - o;
    for (int r = 0; r < b; ++r)
      for (int c = 0; c < b; ++c) (*inv)[(int64_t)X.perm_h[o + r] * n + X.perm_h[o + c]] = h[io + (int64_t)r * b + c];
    io += (int64_t)b * b;
  }
  return GP_OK;
}

namespace {

// Forms the coarsest-level operators at angular frequency w in b, the layout of
// an entry's memory: K^-1, N^-1 G^T, B, the auxiliary inverse.
gp_status coarse_form(const Hierarchy &H, double w, C2<double> *b, hipStream_t s) {
  const int64_t ne = H.neL, nn = H.nnL, na = H.aux.nL;
  TmpArena T;
  struct Free { Arena &a; ~Free() { a.free_all(); } } fr{T};
  C2<double> *nbuf = nullptr;
  GP_TRY(T.alloc(&nbuf, nn * nn));
  C2<double> *pb = b + ne * ne, *bb = pb + ne * nn, *ab = bb + ne * nn;
  if (ne) k_form_freq<<<blocks_for(ne * ne), 256, 0, s>>>(ne * ne, w, H.KLd[0], H.KLd[1], H.KLd[2], b);
  if (nn) {
    k_form_freq<<<blocks_for(nn * nn), 256, 0, s>>>(nn * nn, w, nullptr, H.NLd[0], H.NLd[1], nbuf);
    k_form_freq<<<blocks_for(ne * nn), 256, 0, s>>>(ne * nn, w, nullptr, H.BLd[0], H.BLd[1], bb);
  }
  GP_TRY(dense_inverse_batched(b, (int)ne, 1, s));
  GP_TRY(dense_inverse_batched(nbuf, (int)nn, 1, s));
  if (nn) k_coarse_ng<<<blocks_for(nn * ne), 256, 0, s>>>(nn, ne, nbuf, H.GTLd, pb);
  GP_HIP(hipStreamSynchronize(s));  // nbuf is freed here
  if (na && !H.aux.eig) GP_TRY(aux_coarse_inverse(H.aux, w, ab, s));
  return GP_OK;
}

// A new entry's slot.  The entry joins the cache only once its matrices are
// formed: a call that fails leaves nothing that a later one would find.
gp_status coarse_add(const Hierarchy &H, CoarseCache &C, double w, int32_t *slot, hipStream_t s) {
  const int64_t eb = std::max<int64_t>(coarse_entry_bytes(H), 16);
  GP_TRY(coarse_make_room(C, eb, s));
  void *mem = nullptr;
  if (device_malloc(&mem, (size_t)eb) != hipSuccess) return fail(GP_ERR_NOMEM, "coarse cache entry allocation failed");
  const gp_status st = coarse_form(H, w, (C2<double> *)mem, s);
  if (st != GP_OK) {
    (void)hipStreamSynchronize(s);
    (void)hipFree(mem);
    return st;
  }
  int32_t q = 0;
  while (q < (int32_t)C.e.size() && C.e[q].mem) ++q;
  if (q == (int32_t)C.e.size()) C.e.emplace_back();
  CoarseEntry &x = C.e[q];
  x.omega = w;
  x.mem = mem;
  x.bytes = eb;
  C.bytes += eb;
  C.stale = true;
  *slot = q;
  return GP_OK;
}

}  // namespace

gp_status coarse_cache_lookup(const Hierarchy &H, CoarseCache &C, const std::vector<double> &omegas,
                              std::vector<int32_t> *slots, hipStream_t s, int pin) {
  const auto t0 = std::chrono::steady_clock::now();
  ScratchScope scratch(s);
  slots->assign(omegas.size(), -1);
  if (H.aux.nL > 0 && H.aux.nblk == 0) return fail(GP_ERR_STATE, "auxiliary coarsest level without its block structure");
  // a call that fails keeps no pins
  struct Unpin {
    CoarseCache &c; const std::vector<int32_t> &v; size_t n;
    ~Unpin() { for (size_t i = 0; i < n; ++i) coarse_cache_unpin(c, v[i]); }
  } pins{C, *slots, 0};
  bool fresh = false;
  for (size_t i = 0; i < omegas.size(); ++i) {
    int32_t q = -1;
    for (int32_t t = 0; t < (int32_t)C.e.size(); ++t)
      if (C.e[t].mem && C.e[t].omega == omegas[i]) { q = t; break; }
    if (q < 0) {
      GP_TRY(coarse_add(H, C, omegas[i], &q, s));
      fresh = true;
    }
    C.e[q].used = ++C.clock;
    (*slots)[i] = q;
    if (pin) { ++C.e[q].pins; pins.n = i + 1; }
  }
  if (C.stale || !C.tab) GP_TRY(coarse_table_write(H, C, s));
  pins.n = 0;
  if (fresh) C.form_ms += std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
  return GP_OK;
}

void coarse_cache_unpin(CoarseCache &C, int32_t slot) {
  if (slot >= 0 && slot < (int32_t)C.e.size() && C.e[slot].pins > 0) --C.e[slot].pins;
}

void coarse_cache_free(CoarseCache &C) {
  for (CoarseEntry &x : C.e)
    if (x.mem) (void)hipFree(x.mem);
  if (C.tab) (void)hipFree((void *)C.tab);
  C.e.clear();
  C.tab = nullptr;
  C.cap = 0;
  C.stale = false;
  C.bytes = 0;
}

template <class T>
gp_status vwork_create(gp_layout *lay, const Hierarchy &H, int k, VWork<T> *w) {
  (void)lay;
  Arena &A = w->arena;
  w->k = k;
  GP_TRY(A.alloc(&w->c1, k)); GP_TRY(A.alloc(&w->c2, k)); GP_TRY(A.alloc(&w->fidx, k));
  const size_t nl = H.L.size();
  w->r.assign(nl, nullptr); w->u.assign(nl, nullptr); w->phi.assign(nl, nullptr); w->res.assign(nl, nullptr);
  w->tmp.assign(nl, nullptr); w->rn.assign(nl, nullptr); w->dn.assign(nl, nullptr); w->dn2.assign(nl, nullptr);
  for (size_t l = 0; l < nl; ++l) {
    const int64_t ne = H.L[l].ne * k, nn = H.L[l].nn * k;
    GP_TRY(A.alloc(&w->r[l], ne)); GP_TRY(A.alloc(&w->u[l], ne)); GP_TRY(A.alloc(&w->phi[l], nn));
    GP_TRY(A.alloc(&w->res[l], ne)); GP_TRY(A.alloc(&w->tmp[l], ne)); GP_TRY(A.alloc(&w->rn[l], nn));
    GP_TRY(A.alloc(&w->dn[l], nn)); GP_TRY(A.alloc(&w->dn2[l], nn));
  }
  GP_TRY(A.alloc(&w->crs, std::max<int64_t>((H.neL + H.nnL) * k, 1)));
  const AuxAMG &X = H.aux;
  w->ar.assign(X.L.size(), nullptr); w->ax.assign(X.L.size(), nullptr); w->at.assign(X.L.size(), nullptr);
  for (size_t l = 0; l < X.L.size(); ++l) {
    GP_TRY(A.alloc(&w->ar[l], X.L[l].n * k)); GP_TRY(A.alloc(&w->ax[l], X.L[l].n * k)); GP_TRY(A.alloc(&w->at[l], X.L[l].n * k));
  }
  GP_TRY(A.alloc(&w->a, X.naux * k));
  if (X.eig) GP_TRY(A.alloc(&w->eig_y, X.nL * k));
  GP_TRY(A.alloc(&w->r0, H.L[0].ne * k));
  int64_t nlp = (int64_t)X.GxT.nlong * k, ncp = (int64_t)X.GxT.nchunk * k;
  for (const AuxLevel &L : X.L) {
    nlp = std::max(nlp, (int64_t)L.N.nlong * 2 * k);
    nlp = std::max(nlp, (int64_t)std::max(L.P.nlong, L.PT.nlong) * k);
    ncp = std::max(ncp, (int64_t)L.N.nchunk * 2 * k);
    ncp = std::max(ncp, (int64_t)std::max(L.P.nchunk, L.PT.nchunk) * k);
  }
  GP_TRY(A.alloc(&w->lp, std::max<int64_t>(nlp, 1)));
  GP_TRY(A.alloc(&w->lpart, std::max<int64_t>(ncp, 1)));
  return GP_OK;
}

template <class T>
gp_status vwork_set_columns(VWork<T> &w, const double *omega_cols, const int32_t *fslot_cols, const CoarseCache &C,
                            hipStream_t s) {
  const int k = w.k;
  std::vector<T> c1(k), c2(k);
  for (int j = 0; j < k; ++j) { c1[j] = (T)(-omega_cols[j] * omega_cols[j]); c2[j] = (T)omega_cols[j]; }
  GP_HIP(hipMemcpyAsync(w.c1, c1.data(), sizeof(T) * k, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(w.c2, c2.data(), sizeof(T) * k, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(w.fidx, fslot_cols, sizeof(int32_t) * k, hipMemcpyHostToDevice, s));
  GP_HIP(hipStreamSynchronize(s));  // the host arrays may go out of scope
  w.tab = C.tab;
  w.cap = C.cap;
  return GP_OK;
}

template <class T>
void vwork_free(VWork<T> *w) {
  w->arena.free_all();
}

// ---------------------------------------------------------------- V-cycle kernels

namespace {

template <class T>
__device__ __forceinline__ C2<T> cmul(C2<T> a, C2<T> b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
template <class T>
__device__ __forceinline__ C2<T> cdiv(C2<T> a, C2<T> b) {
  T d = b.x * b.x + b.y * b.y;
  return {(a.x * b.x + a.y * b.y) / d, (a.y * b.x - a.x * b.y) / d};
}

// l1-scaled diagonal: a_ii * (1 + L / |a_ii|), L a bound on the off-diagonal row sum of |a_ij(w)|
template <class T>
__device__ __forceinline__ C2<T> l1diag(C2<T> a, T L) {
  T m = sqrt(a.x * a.x + a.y * a.y);
  T f = m > (T)0 ? (T)1 + L / m : (T)1;
  return {a.x * f, a.y * f};
}

// acc -= a x for a real a, and acc -= (ar + i ai) x, with the fused
// multiply-adds written out: the level-0 edge smoother's two kernels
// (k_edge_sell, k_edge_march) then round alike whatever the compiler would
// fuse in each
template <class T>
__device__ __forceinline__ void csub_re(C2<T> &acc, T a, const C2<T> &x) {
  acc.x = fma(-a, x.x, acc.x);
  acc.y = fma(-a, x.y, acc.y);
}
template <class T>
__device__ __forceinline__ void csub_cx(C2<T> &acc, T ar, T ai, const C2<T> &x) {
  acc.x -= fma(ar, x.x, -(ai * x.y));
  acc.y -= fma(ar, x.y, ai * x.x);
}
// the l1-Jacobi update u + damp * acc / d_l1 of one slot (same reason)
template <class T>
__device__ __forceinline__ C2<T> jacobi_update(const C2<T> &acc, const C2<T> &u0, T c1, T c2, T d0, T d1, T d2, T l0,
                                               T l1, T l2, T damp) {
  const C2<T> dq = l1diag<T>({fma(c1, d1, d0), c2 * d2}, fma(c2, l2, fma(fabs(c1), l1, l0)));
  const C2<T> z = cdiv(acc, dq);
  return {fma(damp, z.x, u0.x), fma(damp, z.y, u0.y)};
}

// Products of the long rows (kLongRow), in two passes.  k_long_part: one block
// per chunk of kLongChunk entries, threads = (column j, entry group g); the
// groups' sums are combined in LDS in a fixed order into
// part[(c*nv + b)*k + j] = sum_{p in chunk c} v_b[p] x[ci[p]][j].
// k_long_fin: lp[(q*nv + b)*k + j] = sum of row q's chunk partials, in order.
template <class T>
__global__ void __launch_bounds__(256) k_long_part(MatV<T> M, int k, const C2<T> *__restrict__ x, C2<T> *__restrict__ part) {
  __shared__ C2<T> red[3][256];
  const int c = blockIdx.x;
  const int tid = threadIdx.x;
  const int j = tid % k, g = tid / k, G = blockDim.x / k;
  C2<T> s[3] = {{0, 0}, {0, 0}, {0, 0}};
  const int64_t pe = M.lce[c];
#pragma unroll 4
  for (int64_t p = M.lcb[c] + g; p < pe; p += G) {
    const C2<T> xv = x[(int64_t)M.ci[p] * k + j];
    for (int b = 0; b < M.nv; ++b) {
      const T a = M.v[b][p];
      s[b].x += a * xv.x;
      s[b].y += a * xv.y;
    }
  }
  for (int b = 0; b < M.nv; ++b) red[b][tid] = s[b];
  __syncthreads();
  if (tid < k) {
    for (int b = 0; b < M.nv; ++b) {
      C2<T> t = {0, 0};
      for (int gg = 0; gg < G; ++gg) { t.x += red[b][gg * k + j].x; t.y += red[b][gg * k + j].y; }
      part[((int64_t)c * M.nv + b) * k + j] = t;
    }
  }
}

// one block per long row: thread (bj, g) sums chunks g, g + G, ... of row q
// for output bj = b*k + j; the G partial sums are combined in LDS in order
template <class T>
__global__ void __launch_bounds__(256) k_long_fin(MatV<T> M, int k, const C2<T> *__restrict__ part, C2<T> *__restrict__ lp) {
  __shared__ C2<T> red[256];
  const int q = blockIdx.x;
  const int per = M.nv * k;  // <= 128 (nv <= 2, k <= 64)
  const int tid = threadIdx.x;
  const int bj = tid % per, g = tid / per, G = blockDim.x / per;
  C2<T> acc = {0, 0};
  if (g < G)
    for (int c = M.lqp[q] + g; c < M.lqp[q + 1]; c += G) {
      const C2<T> v = part[(int64_t)c * per + bj];
      acc.x += v.x;
      acc.y += v.y;
    }
  red[tid] = acc;
  __syncthreads();
  if (tid < per) {
    C2<T> t = {0, 0};
    for (int gg = 0; gg < G; ++gg) { t.x += red[gg * per + tid].x; t.y += red[gg * per + tid].y; }
    lp[(int64_t)q * per + tid] = t;
  }
}

// NOK (or-ed into RES or JACOBI): r already holds a residual with the K(w) u
// term for the current u, so only B(w) phi is subtracted; phi is then the
// change of the nodal iterate since r was formed.
struct EdgeMode { enum { RES = 0, JACOBI = 1, JACOBI0 = 2, KIND = 3, NOK = 4 }; };

// Edge kernel, one thread per (row, column):
//   acc = r - K(w) u - B(w) phi           (without K(w) u under NOK)
//   RES:     res = acc
//   JACOBI:  u_out = u + acc / d_l1
//   JACOBI0: u_out = r / d_l1           (u = phi = 0)
template <class T>
__global__ void k_edge(int64_t nr, int k, MatV<T> K, MatV<T> B, const T *__restrict__ c1v, const T *__restrict__ c2v,
                       const T *__restrict__ kd0, const T *__restrict__ kd1, const T *__restrict__ kd2,
                       const T *__restrict__ kl0, const T *__restrict__ kl1, const T *__restrict__ kl2,
                       const C2<T> *__restrict__ r, const C2<T> *__restrict__ u, const C2<T> *__restrict__ phi,
                       C2<T> *__restrict__ out, int mode, int use_phi, T damp) {
  int64_t t = xcd_block_id() * blockDim.x + threadIdx.x;
  int64_t i = t / k;
  int j = (int)(t - i * k);
  if (i >= nr) return;
  const T c1 = c1v[j], c2 = c2v[j];
  C2<T> acc = r[i * k + j];
  const int kind = mode & EdgeMode::KIND;
  if (kind != EdgeMode::JACOBI0) {
    if (mode & EdgeMode::NOK) {
    } else if (K.dg[0]) {  // K_eps and K_sig diagonal (level 0): one value array in the loop
      for (int64_t p = K.rp[i]; p < K.rp[i + 1]; ++p) {
        const T a = K.v[0][p];
        const C2<T> x = u[(int64_t)K.ci[p] * k + j];
        acc.x -= a * x.x;
        acc.y -= a * x.y;
      }
      const C2<T> a = {c1 * K.dg[0][i], c2 * K.dg[1][i]};
      const C2<T> x = u[i * k + j];
      acc.x -= a.x * x.x - a.y * x.y;
      acc.y -= a.x * x.y + a.y * x.x;
    } else
    for (int64_t p = K.rp[i]; p < K.rp[i + 1]; ++p) {
      C2<T> a = {K.v[0][p] + c1 * K.v[1][p], c2 * K.v[2][p]};
      C2<T> x = u[(int64_t)K.ci[p] * k + j];
      acc.x -= a.x * x.x - a.y * x.y;
      acc.y -= a.x * x.y + a.y * x.x;
    }
    if (use_phi) {
      for (int64_t p = B.rp[i]; p < B.rp[i + 1]; ++p) {
        C2<T> b = {c1 * B.v[0][p], c2 * B.v[1][p]};
        C2<T> x = phi[(int64_t)B.ci[p] * k + j];
        acc.x -= b.x * x.x - b.y * x.y;
        acc.y -= b.x * x.y + b.y * x.x;
      }
    }
  }
  if (kind == EdgeMode::RES) { out[i * k + j] = acc; return; }
  C2<T> d = l1diag<T>({kd0[i] + c1 * kd1[i], c2 * kd2[i]}, kl0[i] + fabs(c1) * kl1[i] + c2 * kl2[i]);
  C2<T> q = cdiv(acc, d);
  if (kind == EdgeMode::JACOBI0) { out[i * k + j] = {damp * q.x, damp * q.y}; return; }
  C2<T> u0 = u[i * k + j];
  out[i * k + j] = {u0.x + damp * q.x, u0.y + damp * q.y};
}

// Level-0 edge smoother / residual on the sliced-ELL K and B.  LPR adjacent
// lanes share one row and each holds SPL consecutive slots (one 16-byte load
// per gathered neighbour row), so one wave-wide gather touches the lines of
// 64 / LPR rows, not 64: with one thread per row and all slots in registers
// the L1 tag lookups of the scattered 16-byte pieces, not HBM, set the pace.
// Walks the SELL row at slice base b0 / width wd / lane with four row
// gathers in flight per lane: batches of 4 entries, then single entries
// (batches of 8 ran slower: 687 vs 536 us for the level-0 edge smoother,
// register pressure); each batch reads its indices and values first, then its
// gathered rows of x, and calls f(a0, a1, a2, xrow) for every entry in
// order (one dependent index -> row chain per entry left these kernels
// latency-bound).
template <class T, int KS, int NV, int NB, int ES, class F>
__device__ __forceinline__ void sell_batch(const SellV<T> &M, int64_t b0, int t0, int lane, const C2<T> *__restrict__ x,
                                           int k, int j0, F &f) {
  int32_t c[NB];
  T a[NV][NB];
#pragma unroll
  for (int h = 0; h < NB; ++h) {
    const int64_t e = b0 + (int64_t)(t0 + h * ES) * 64 + lane;
    // plain loads: a small operator then stays in L2 from one launch to the next
    // (edge launches of a 60x20x8 layout 7.0 us with non-temporal loads, 5.4 with
    // these; 9.0 and 7.2 at 48x48x12 in FP64), and where the operator streams
    // the gathered rows of x keep their places all the same (level 0 at
    // 200x200x24 224 us either way, a 400x400x32 solve 2286 and 2267 ms)
    c[h] = M.ci[e];
#pragma unroll
    for (int v = 0; v < NV; ++v) a[v][h] = M.v[v][e];
  }
  C2<T> xv[NB][KS];
#pragma unroll
  for (int h = 0; h < NB; ++h) load_slots<T, KS>(x + (int64_t)c[h] * k + j0, xv[h]);
#pragma unroll
  for (int h = 0; h < NB; ++h)
    f(a[0][h], NV > 1 ? a[NV > 1 ? 1 : 0][h] : T(0), NV > 2 ? a[NV > 2 ? 2 : 0][h] : T(0), xv[h]);
}

template <class T, int KS, int NV, class F>
__device__ __forceinline__ void sell_row(const SellV<T> &M, int64_t b0, int wd, int lane, const C2<T> *__restrict__ x,
                                         int k, int j0, F &&f) {
  int t0 = 0;
  for (; t0 + 4 <= wd; t0 += 4) sell_batch<T, KS, NV, 4, 1>(M, b0, t0, lane, x, k, j0, f);
  for (; t0 < wd; ++t0) sell_batch<T, KS, NV, 1, 1>(M, b0, t0, lane, x, k, j0, f);
}

// Entry-split walk: the lane group es of ES groups sharing a row takes the
// entries es, es + ES, es + 2 ES, ... (see entry_split).  es_reduce then sums
// the groups' partial results: the groups of a row sit LPR lanes apart inside an
// aligned LPR*ES-lane block of the wavefront, so xor shuffles over LPR, 2 LPR,
// ... stay inside the row.
template <class T, int KS, int NV, int ES, class F>
__device__ __forceinline__ void sell_row_es(const SellV<T> &M, int64_t b0, int wd, int lane, int es,
                                            const C2<T> *__restrict__ x, int k, int j0, F &&f) {
  if (ES == 1) { sell_row<T, KS, NV>(M, b0, wd, lane, x, k, j0, f); return; }
  int t0 = es;
  for (; t0 + 3 * ES < wd; t0 += 4 * ES) sell_batch<T, KS, NV, 4, ES>(M, b0, t0, lane, x, k, j0, f);
  for (; t0 < wd; t0 += ES) sell_batch<T, KS, NV, 1, ES>(M, b0, t0, lane, x, k, j0, f);
}

template <class T, int KS, int LPR, int ES>
__device__ __forceinline__ void es_reduce(C2<T> (&acc)[KS]) {
#pragma unroll
  for (int m = LPR; m < LPR * ES; m <<= 1)
#pragma unroll
    for (int q = 0; q < KS; ++q) { acc[q].x += __shfl_xor(acc[q].x, m); acc[q].y += __shfl_xor(acc[q].y, m); }
}

template <class T, int SPL, int LPR>
__global__ void __launch_bounds__(256) k_edge_sell(int64_t nr, int k, SellV<T> K, SellV<T> B, const T *__restrict__ c1v,
                                                   const T *__restrict__ c2v, const T *__restrict__ kd0,
                                                   const T *__restrict__ kd1, const T *__restrict__ kd2,
                                                   const T *__restrict__ kl0, const T *__restrict__ kl1,
                                                   const T *__restrict__ kl2, const C2<T> *__restrict__ r,
                                                   const C2<T> *__restrict__ u, const C2<T> *__restrict__ phi,
                                                   C2<T> *__restrict__ out, int mode, int use_phi, T damp) {
  constexpr int KS = SPL;
  const int64_t t = xcd_block_id() * blockDim.x + threadIdx.x;
  const int64_t pos = t / LPR;
  if (pos >= nr) return;
  const int sub = (int)(t - pos * LPR);
  const int64_t i = K.rows ? (int64_t)K.rows[pos] : pos;  // B shares K's slot order
  const int j0 = ((int)blockIdx.y * LPR + sub) * SPL;
  const int64_t sl = pos >> 6;
  const int lane = (int)(pos & 63);
  T c1[KS], c2[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) { c1[q] = c1v[j0 + q]; c2[q] = c2v[j0 + q]; }
  C2<T> acc[KS];
  load_slots<T, KS>(r + i * k + j0, acc);
  const int kind = mode & EdgeMode::KIND;
  if (kind != EdgeMode::JACOBI0 && !(mode & EdgeMode::NOK)) {
    const int64_t b0 = K.base[sl];
    const int wd = K.w[sl];
    if (K.nv == 1) {
      sell_row<T, KS, 1>(K, b0, wd, lane, u, k, j0, [&](T a, T, T, const C2<T>(&x)[KS]) {
#pragma unroll
        for (int q = 0; q < KS; ++q) csub_re<T>(acc[q], a, x[q]);
      });
    } else {
      sell_row<T, KS, 3>(K, b0, wd, lane, u, k, j0, [&](T a0, T a1, T a2, const C2<T>(&x)[KS]) {
#pragma unroll
        for (int q = 0; q < KS; ++q) {
          const T ar = a0 + c1[q] * a1, ai = c2[q] * a2;
          acc[q].x -= ar * x[q].x - ai * x[q].y;
          acc[q].y -= ar * x[q].y + ai * x[q].x;
        }
      });
    }
    if (K.dg[0]) {  // diagonal K_eps, K_sig (and K_S when kept out of the entries)
      const T de = K.dg[0][i], ds = K.dg[1][i];
      C2<T> x[KS];
      load_slots<T, KS>(u + i * k + j0, x);
      if (K.dgs) {
        const T dsg = K.dgs[i];
#pragma unroll
        for (int q = 0; q < KS; ++q) csub_cx<T>(acc[q], fma(c1[q], de, dsg), c2[q] * ds, x[q]);
      } else {
#pragma unroll
        for (int q = 0; q < KS; ++q) csub_cx<T>(acc[q], c1[q] * de, c2[q] * ds, x[q]);
      }
    }
  }
  if (kind != EdgeMode::JACOBI0) {
    if (use_phi) {
      sell_row<T, KS, 2>(B, B.base[sl], B.w[sl], lane, phi, k, j0, [&](T a0, T a1, T, const C2<T>(&x)[KS]) {
#pragma unroll
        for (int q = 0; q < KS; ++q) csub_cx<T>(acc[q], c1[q] * a0, c2[q] * a1, x[q]);
      });
    }
  }
  if (kind == EdgeMode::RES) { store_slots<T, KS>(out + i * k + j0, acc); return; }
  const T d0 = kd0[i], d1 = kd1[i], d2 = kd2[i], l0 = kl0[i], l1 = kl1[i], l2 = kl2[i];
  C2<T> u0[KS];
  if (kind == EdgeMode::JACOBI) load_slots<T, KS>(u + i * k + j0, u0);
  else
#pragma unroll
    for (int q = 0; q < KS; ++q) u0[q] = {(T)0, (T)0};
#pragma unroll
  for (int q = 0; q < KS; ++q) acc[q] = jacobi_update<T>(acc[q], u0[q], c1[q], c2[q], d0, d1, d2, l0, l1, l2, damp);
  store_slots<T, KS>(out + i * k + j0, acc);
}

// The edge launches that gather no K u (NOK: r - B phi, and the Jacobi
// sweep from such a residual; JACOBI0: r / d_l1) stream r and out and gather
// two phi rows per edge.  They were bound by the bytes in flight, not by the
// texture path's rate: here each lane group takes two rows (positions p and
// p + half), whose residual, B indices and values, diagonals and u are all
// loaded before either row's phi gathers.  Per row the same operations in
// the same order as k_edge_sell.  The matrix loads are non-temporal here, in
// k_spmv2_sell2 and in the march: such operators stream past every cache (a
// 400x400x32 step 2227 ms with them, 2225 with plain loads; runs of one side
// differ by 1 %).
constexpr int64_t kNok2MinRows = (int64_t)1 << 22;

template <class T, int SPL, int LPR>
__global__ void __launch_bounds__(256) k_edge_nok2(int64_t nr, int64_t half, int k, SellV<T> K, SellV<T> B,
                                                   const T *__restrict__ c1v, const T *__restrict__ c2v,
                                                   const T *__restrict__ kd0, const T *__restrict__ kd1,
                                                   const T *__restrict__ kd2, const T *__restrict__ kl0,
                                                   const T *__restrict__ kl1, const T *__restrict__ kl2,
                                                   const C2<T> *__restrict__ r, const C2<T> *__restrict__ u,
                                                   const C2<T> *__restrict__ phi, C2<T> *__restrict__ out, int mode,
                                                   int use_phi, T damp) {
  constexpr int KS = SPL, NR = 2, PFB = 2;
  const int64_t t = xcd_block_id() * blockDim.x + threadIdx.x;
  const int64_t q0 = t / LPR;
  if (q0 >= half) return;
  const int sub = (int)(t - q0 * LPR);
  const int j0 = ((int)blockIdx.y * LPR + sub) * SPL;
  const int kind = mode & EdgeMode::KIND;
  const bool bphi = use_phi && kind != EdgeMode::JACOBI0;
  T c1[KS], c2[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) { c1[q] = c1v[j0 + q]; c2[q] = c2v[j0 + q]; }
  bool ok[NR];
  int64_t i[NR], bb[NR];
  int wb[NR], lane[NR];
  C2<T> acc[NR][KS], u0[NR][KS];
  T d[NR][6];
  int32_t cb[NR][PFB];
  T a0[NR][PFB], a1[NR][PFB];
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    const int64_t pos = q0 + n * half;
    ok[n] = pos < nr;
    i[n] = 0; bb[n] = 0; wb[n] = 0; lane[n] = 0;
    if (!ok[n]) continue;
    i[n] = K.rows ? (int64_t)K.rows[pos] : pos;
    const int64_t sl = pos >> 6;
    lane[n] = (int)(pos & 63);
    if (bphi) { bb[n] = B.base[sl]; wb[n] = B.w[sl]; }
  }
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    if (!ok[n]) continue;
    load_slots<T, KS>(r + i[n] * k + j0, acc[n]);
    if (kind != EdgeMode::RES) {
      d[n][0] = kd0[i[n]]; d[n][1] = kd1[i[n]]; d[n][2] = kd2[i[n]];
      d[n][3] = kl0[i[n]]; d[n][4] = kl1[i[n]]; d[n][5] = kl2[i[n]];
    }
    if (kind == EdgeMode::JACOBI) load_slots<T, KS>(u + i[n] * k + j0, u0[n]);
    else
#pragma unroll
      for (int q = 0; q < KS; ++q) u0[n][q] = {(T)0, (T)0};
#pragma unroll
    for (int h = 0; h < PFB; ++h) {
      cb[n][h] = 0; a0[n][h] = (T)0; a1[n][h] = (T)0;
      if (h < wb[n]) {
        const int64_t e = bb[n] + (int64_t)h * 64 + lane[n];
        cb[n][h] = __builtin_nontemporal_load(B.ci + e);
        a0[n][h] = __builtin_nontemporal_load(B.v[0] + e);
        a1[n][h] = __builtin_nontemporal_load(B.v[1] + e);
      }
    }
  }
  C2<T> xb[NR][PFB][KS];
#pragma unroll
  for (int n = 0; n < NR; ++n)
#pragma unroll
    for (int h = 0; h < PFB; ++h)
      if (h < wb[n]) load_slots<T, KS>(phi + (int64_t)cb[n][h] * k + j0, xb[n][h]);
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    if (!ok[n]) continue;
#pragma unroll
    for (int h = 0; h < PFB; ++h)
      if (h < wb[n])
#pragma unroll
        for (int q = 0; q < KS; ++q) csub_cx<T>(acc[n][q], c1[q] * a0[n][h], c2[q] * a1[n][h], xb[n][h][q]);
    auto fb = [&](T b0v, T b1v, T, const C2<T>(&x)[KS]) {
#pragma unroll
      for (int q = 0; q < KS; ++q) csub_cx<T>(acc[n][q], c1[q] * b0v, c2[q] * b1v, x[q]);
    };
    for (int tt = PFB; tt < wb[n]; ++tt) sell_batch<T, KS, 2, 1, 1>(B, bb[n], tt, lane[n], phi, k, j0, fb);
    if (kind != EdgeMode::RES)
#pragma unroll
      for (int q = 0; q < KS; ++q)
        acc[n][q] = jacobi_update<T>(acc[n][q], u0[n][q], c1[q], c2[q], d[n][0], d[n][1], d[n][2], d[n][3], d[n][4],
                                     d[n][5], damp);
    store_slots<T, KS>(out + i[n] * k + j0, acc[n]);
  }
}

// ---- level-0 edge smoother / residual as a plane march (FP32) --------------
// k_edge_sell with the K u gathers served from LDS.  A workgroup takes one
// (tile half, run of planes, group of SW slots) and walks its planes upwards
// holding u of planes z - 1, z, z + 1 (the rows of blocks (tile, plane,
// half), SW slots each) in a ring of three LDS plane buffers.  Each row's
// couplings lie in those three blocks except at the tile half's sides
// (code[e] < 0: read from global memory as in k_edge_sell).  The next plane's
// u is loaded into registers while the current plane is computed and written
// to LDS after it, and each thread computes its rows of a plane together, so
// the dependent loads of both rows are in flight at once.  Entries are summed
// in k_edge_sell's order with the same operations: both kernels give the same
// bits.
constexpr int kMarchThreads = 768;
constexpr int kMarchPlanes = 11;                       // planes per run (a run stages one more on each side)
constexpr int kMarchMaxRows = kMarchHalf * kTile * 3;  // rows of one block: 8 ix x 16 iy x 3 directions

// u of slots [jl, jl + 4) of LDS row off in ring buffer slot; swap reads the
// two 16-byte halves in the other order (rows of alternate lane quads then
// touch disjoint LDS banks in each read)
template <int SW>
__device__ __forceinline__ void march_lds_row(const float4 *__restrict__ lds, int slot, int maxb, int off, int jl,
                                              bool swp, C2<float> (&x)[4]) {
  const float4 *q = lds + ((int64_t)slot * maxb + off) * (SW / 2) + (jl >> 1);
  float4 v0, v1;
  if (swp) { v1 = q[1]; v0 = q[0]; } else { v0 = q[0]; v1 = q[1]; }
  x[0] = {v0.x, v0.y}; x[1] = {v0.z, v0.w}; x[2] = {v1.x, v1.y}; x[3] = {v1.z, v1.w};
}

template <int LPR>
__global__ void __launch_bounds__(kMarchThreads)
    k_edge_march(int k, int nplane, int zchunk, int nzc, int ngroup, int maxb, const int32_t *__restrict__ start,
                 const int32_t *__restrict__ code, SellV<float> K, SellV<float> B, const float *__restrict__ c1v,
                 const float *__restrict__ c2v, const float *__restrict__ kd0, const float *__restrict__ kd1,
                 const float *__restrict__ kd2, const float *__restrict__ kl0, const float *__restrict__ kl1,
                 const float *__restrict__ kl2, const C2<float> *__restrict__ r, const C2<float> *__restrict__ u,
                 const C2<float> *__restrict__ phi, C2<float> *__restrict__ out, int mode, int use_phi, float damp) {
  constexpr int SPL = 4, SW = LPR * SPL, PR = SW / 2, MT = kMarchThreads, RPP = MT / LPR;
  constexpr int NR = (kMarchMaxRows + RPP - 1) / RPP;       // rows per thread and plane
  constexpr int NQ = (kMarchMaxRows * PR + MT - 1) / MT;   // 16-byte pieces per thread and plane
  extern __shared__ float4 lds[];                          // [3][maxb][PR]
  const int64_t wg = xcd_block_id();
  const int g = (int)(wg % ngroup);
  const int64_t rest = wg / ngroup;
  const int zc = (int)(rest % nzc);
  const int64_t th = rest / nzc;
  const int64_t tile = th >> 1;
  const int half = (int)(th & 1);
  const int z0 = zc * zchunk, z1 = min(z0 + zchunk, nplane);
  if (z0 >= nplane) return;  // the whole workgroup leaves together
  const int tid = (int)threadIdx.x;
  const int sub = tid % LPR, jl = sub * SPL, j0 = g * SW + jl;
  const bool swp = LPR == 4 && ((tid >> 2) & 1);
  float c1[SPL], c2[SPL];
#pragma unroll
  for (int q = 0; q < SPL; ++q) { c1[q] = c1v[j0 + q]; c2[q] = c2v[j0 + q]; }
  const int kind = mode & EdgeMode::KIND;
  const C2<float> *usrc = u + g * SW;

  // u of block (tile, p, half): fetch into registers, put into ring slot p % 3
  auto fetch = [&](int p, float4 (&v)[NQ]) {
    const int64_t b = (tile * nplane + p) * 2 + half;
    const int st = start[b], tot = (start[b + 1] - st) * PR;
#pragma unroll
    for (int a = 0; a < NQ; ++a) {
      const int q = a * MT + tid;
      v[a] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (q < tot) {
        const int row = q / PR, part = q - row * PR;
        v[a] = reinterpret_cast<const float4 *>(usrc + (int64_t)K.rows[st + row] * k)[part];
      }
    }
  };
  auto put = [&](int p, const float4 (&v)[NQ]) {
    const int64_t b = (tile * nplane + p) * 2 + half;
    const int tot = (start[b + 1] - start[b]) * PR;
    float4 *dst = lds + (int64_t)(p % 3) * maxb * PR;
#pragma unroll
    for (int a = 0; a < NQ; ++a) {
      const int q = a * MT + tid;
      if (q < tot) dst[q] = v[a];
    }
  };

  float4 pf[NQ];
  {
    float4 pb[NQ];
    if (z0 > 0) fetch(z0 - 1, pb);
    fetch(z0, pf);
    if (z0 > 0) put(z0 - 1, pb);
    put(z0, pf);
  }
  if (z0 + 1 < nplane) fetch(z0 + 1, pf);
  for (int z = z0; z < z1; ++z) {
    if (z + 1 < nplane) put(z + 1, pf);  // ring slot of plane z - 2, done with since the last barrier
    __syncthreads();
    if (z + 2 < nplane && z + 2 <= z1) fetch(z + 2, pf);  // in flight while plane z is computed
    const int64_t b = (tile * nplane + z) * 2 + half;
    const int st = start[b], m = start[b + 1] - st;
    const int zm1 = z - 1;

    int rr[NR], wd[NR], wb[NR], lane[NR];
    int64_t i[NR], b0[NR], bb[NR];
    bool ok[NR];
    C2<float> acc[NR][SPL];
    int wmax = 0, wbmax = 0;
#pragma unroll
    for (int n = 0; n < NR; ++n) {
      rr[n] = tid / LPR + n * RPP;
      ok[n] = rr[n] < m;
      wd[n] = 0; wb[n] = 0; i[n] = 0; b0[n] = 0; bb[n] = 0; lane[n] = 0;
      if (ok[n]) {
        const int64_t pos = st + rr[n];
        const int64_t sl = pos >> 6;
        lane[n] = (int)(pos & 63);
        i[n] = K.rows[pos];
        b0[n] = K.base[sl];
        wd[n] = K.w[sl];
        if (use_phi) { bb[n] = B.base[sl]; wb[n] = B.w[sl]; }
        load_slots<float, SPL>(r + i[n] * k + j0, acc[n]);
      }
      wmax = max(wmax, wd[n]);
      wbmax = max(wbmax, wb[n]);
    }
    // K u: two entries of each row in flight per round, each row in entry order
    for (int t0 = 0; t0 < wmax; t0 += 2) {
      int32_t c[NR][2];
      float a[NR][2];
#pragma unroll
      for (int n = 0; n < NR; ++n)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          c[n][h] = 0; a[n][h] = 0.f;
          if (t0 + h < wd[n]) {
            const int64_t e = b0[n] + (int64_t)(t0 + h) * 64 + lane[n];
            c[n][h] = __builtin_nontemporal_load(code + e);
            a[n][h] = __builtin_nontemporal_load(K.v[0] + e);
          }
        }
      C2<float> xv[NR][2][SPL];
#pragma unroll
      for (int n = 0; n < NR; ++n)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (t0 + h < wd[n]) {
            if (c[n][h] < 0) load_slots<float, SPL>(u + (int64_t)(c[n][h] & 0x7fffffff) * k + j0, xv[n][h]);
            else march_lds_row<SW>(lds, (zm1 + (c[n][h] >> 16)) % 3, maxb, c[n][h] & 0xffff, jl, swp, xv[n][h]);
          }
        }
#pragma unroll
      for (int n = 0; n < NR; ++n)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (t0 + h < wd[n])
#pragma unroll
            for (int q = 0; q < SPL; ++q) csub_re<float>(acc[n][q], a[n][h], xv[n][h][q]);
    }
    // diagonal K_eps, K_sig with the row's own u (plane z's block, offset rr)
    C2<float> self[NR][SPL];
#pragma unroll
    for (int n = 0; n < NR; ++n)
      if (ok[n]) {
        march_lds_row<SW>(lds, z % 3, maxb, rr[n], jl, swp, self[n]);
        if (K.dg[0]) {
          const float de = K.dg[0][i[n]], ds = K.dg[1][i[n]];
          if (K.dgs) {
            const float dsg = K.dgs[i[n]];
#pragma unroll
            for (int q = 0; q < SPL; ++q) csub_cx<float>(acc[n][q], fmaf(c1[q], de, dsg), c2[q] * ds, self[n][q]);
          } else {
#pragma unroll
            for (int q = 0; q < SPL; ++q) csub_cx<float>(acc[n][q], c1[q] * de, c2[q] * ds, self[n][q]);
          }
        }
      }
    // B phi, each row in entry order
    for (int t = 0; t < wbmax; ++t) {
      float a0[NR], a1[NR];
      int32_t cb[NR];
#pragma unroll
      for (int n = 0; n < NR; ++n) {
        a0[n] = 0.f; a1[n] = 0.f; cb[n] = 0;
        if (t < wb[n]) {
          const int64_t e = bb[n] + (int64_t)t * 64 + lane[n];
          cb[n] = __builtin_nontemporal_load(B.ci + e);
          a0[n] = __builtin_nontemporal_load(B.v[0] + e);
          a1[n] = __builtin_nontemporal_load(B.v[1] + e);
        }
      }
      C2<float> xb[NR][SPL];
#pragma unroll
      for (int n = 0; n < NR; ++n)
        if (t < wb[n]) load_slots<float, SPL>(phi + (int64_t)cb[n] * k + j0, xb[n]);
#pragma unroll
      for (int n = 0; n < NR; ++n)
        if (t < wb[n])
#pragma unroll
          for (int q = 0; q < SPL; ++q) csub_cx<float>(acc[n][q], c1[q] * a0[n], c2[q] * a1[n], xb[n][q]);
    }
#pragma unroll
    for (int n = 0; n < NR; ++n) {
      if (!ok[n]) continue;
      if (kind == EdgeMode::JACOBI) {
        const float d0 = kd0[i[n]], d1 = kd1[i[n]], d2 = kd2[i[n]], l0 = kl0[i[n]], l1 = kl1[i[n]], l2 = kl2[i[n]];
#pragma unroll
        for (int q = 0; q < SPL; ++q)
          acc[n][q] = jacobi_update<float>(acc[n][q], self[n][q], c1[q], c2[q], d0, d1, d2, l0, l1, l2, damp);
      }
      store_slots<float, SPL>(out + i[n] * k + j0, acc[n]);
    }
    __syncthreads();
  }
}

// The march for one level-0 launch that gathers K u (RES or JACOBI without
// NOK) with FP32 data and k a multiple of 8; false when it does not apply or
// the device cannot give the workgroup its LDS (the caller then launches
// k_edge_sell).
bool edge_march(const Hierarchy &H, int k, const SellV<float> &K, const SellV<float> &B, const float *c1,
                const float *c2, const float *kd0, const float *kd1, const float *kd2, const float *kl0,
                const float *kl1, const float *kl2, const C2<float> *r, const C2<float> *u, const C2<float> *phi,
                C2<float> *out, int mode, int use_phi, float damp, hipStream_t s) {
  const EdgeMarch &M = H.march;
  const int kind = mode & EdgeMode::KIND;
  if (!M.code || !u || kind == EdgeMode::JACOBI0 || (mode & EdgeMode::NOK) || k % 8 || K.nv != 1 || !K.rows) return false;
  const int lds_max = M.lds_max;
  const int sw = (k % 16 == 0 && (int64_t)3 * M.maxb * 16 * 8 <= lds_max) ? 16 : 8;
  const int64_t shm = (int64_t)3 * M.maxb * sw * 8;
  if (shm > lds_max || M.maxb == 0 || M.maxb > kMarchMaxRows) return false;
  const int ngroup = k / sw;
  const int nzc = (M.nplane + kMarchPlanes - 1) / kMarchPlanes;
  const int zchunk = (M.nplane + nzc - 1) / nzc;
  const int64_t nwg = M.ntile * 2 * nzc * ngroup;
  if (nwg >= ((int64_t)1 << 31)) return false;
  if (sw == 16) {
    k_edge_march<4><<<(unsigned)nwg, kMarchThreads, (size_t)shm, s>>>(
        k, M.nplane, zchunk, nzc, ngroup, M.maxb, M.start, M.code, K, B, c1, c2, kd0, kd1, kd2, kl0, kl1, kl2, r, u,
        phi, out, mode, use_phi, damp);
  } else {
    k_edge_march<2><<<(unsigned)nwg, kMarchThreads, (size_t)shm, s>>>(
        k, M.nplane, zchunk, nzc, ngroup, M.maxb, M.start, M.code, K, B, c1, c2, kd0, kd1, kd2, kl0, kl1, kl2, r, u,
        phi, out, mode, use_phi, damp);
  }
  return true;
}

// SELL nodal l1-Jacobi sweep (contract of k_node, d given) of an operator without listed rows
template <class T, int SPL, int LPR, int ES>
__global__ void __launch_bounds__(256) k_node_sell(int64_t nr, int k, SellV<T> N, const T *__restrict__ c1v,
                                                   const T *__restrict__ c2v, const T *__restrict__ nd0,
                                                   const T *__restrict__ nd1, const T *__restrict__ nl0,
                                                   const T *__restrict__ nl1, const C2<T> *__restrict__ rn,
                                                   const C2<T> *__restrict__ d, C2<T> *__restrict__ dout, T damp) {
  constexpr int KS = SPL;  // LPR adjacent lanes share a row, SPL slots each;
                           // ES such groups split the row's entries
  const int64_t t_ = xcd_block_id() * blockDim.x + threadIdx.x;
  const int64_t pos = t_ / (LPR * ES);
  if (pos >= nr) return;
  const int sub = (int)(t_ - pos * (LPR * ES)), es = sub / LPR;
  const int j0 = ((int)blockIdx.y * LPR + (sub - es * LPR)) * SPL;
  const int64_t i = N.rows ? (int64_t)N.rows[pos] : pos;  // slot position -> row
  T c1[KS], c2[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) { c1[q] = c1v[j0 + q]; c2[q] = c2v[j0 + q]; }
  C2<T> acc[KS];
  if (es == 0) load_slots<T, KS>(rn + i * k + j0, acc);
  else
#pragma unroll
    for (int q = 0; q < KS; ++q) acc[q] = {0, 0};
  {
    const int64_t sl = pos >> 6;
    const int lane = (int)(pos & 63);
    const int64_t b0 = N.base[sl];
    const int wd = N.w[sl];
    sell_row_es<T, KS, 2, ES>(N, b0, wd, lane, es, d, k, j0, [&](T a0, T a1, T, const C2<T>(&x)[KS]) {
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        const T ar = c1[q] * a0, ai = c2[q] * a1;
        acc[q].x -= ar * x[q].x - ai * x[q].y;
        acc[q].y -= ar * x[q].y + ai * x[q].x;
      }
    });
  }
  es_reduce<T, KS, LPR, ES>(acc);
  if (es != 0) return;
  const T e0 = nd0[i], e1 = nd1[i], m0 = nl0[i], m1 = nl1[i];
  C2<T> o[KS];
  load_slots<T, KS>(d + i * k + j0, o);
#pragma unroll
  for (int q = 0; q < KS; ++q) {
    const C2<T> dg = l1diag<T>({c1[q] * e0, c2[q] * e1}, fabs(c1[q]) * m0 + c2[q] * m1);
    const C2<T> z = cdiv(acc[q], dg);
    o[q] = {o[q].x + damp * z.x, o[q].y + damp * z.y};
  }
  store_slots<T, KS>(dout + i * k + j0, o);
}

// Optional epilogues of the products that form a right-hand side, taken while it
// is in registers instead of by a pass of its own.  Jac0, over edge rows y:
// u = damp y / d_l1, the edge smoother's first sweep from zero.
template <class T>
struct Jac0 {
  const T *kd0 = nullptr, *kd1 = nullptr, *kd2 = nullptr, *kl0 = nullptr, *kl1 = nullptr, *kl2 = nullptr;
  C2<T> *u = nullptr;
  T damp = (T)1;
};
template <class T, int KS>
__device__ __forceinline__ void jac0_store(const Jac0<T> &jz, int64_t i, int k, int j0, const T (&c1)[KS], const T (&c2)[KS],
                                           const C2<T> (&o)[KS]) {
  const T d0 = jz.kd0[i], d1 = jz.kd1[i], d2 = jz.kd2[i], l0 = jz.kl0[i], l1 = jz.kl1[i], l2 = jz.kl2[i];
  C2<T> uo[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) {
    const C2<T> dq = l1diag<T>({d0 + c1[q] * d1, c2[q] * d2}, l0 + fabs(c1[q]) * l1 + c2[q] * l2);
    const C2<T> z = cdiv(o[q], dq);
    uo[q] = {jz.damp * z.x, jz.damp * z.y};
  }
  store_slots<T, KS>(jz.u + i * k + j0, uo);
}
// Nod0, over nodal rows y = G^T res: d = damp y / d_n, the nodal smoother's first
// sweep from zero, and with sum also sum += d.  y itself is stored only where a
// second sweep reads it.
template <class T>
struct Nod0 {
  const T *nd0 = nullptr, *nd1 = nullptr, *nl0 = nullptr, *nl1 = nullptr;
  C2<T> *d = nullptr, *sum = nullptr;
  T damp = (T)1;
};

// SELL y = M x (real M) or y += M x, an operator without listed rows; EP names
// the epilogue.  One level's edge and nodal prolongations share a launch
// (k_prolong_sell).  Most of a small level's launch is the launch (2.5-6 us at
// 48x48x12), and a level of the edge V-cycle takes 9 of them now instead of 14;
// on large levels the passes over rn and phi go.  Solve of a 60x20x8 layout 10.1
// -> 9.2 ms, 48x48x12 in FP64 18.2 -> 16.8, 8 ports at 128x128x16 164.0 -> 157.5,
// at 200x200x24 333.3 -> 324.9.
enum SpmvEp { SPMV_PLAIN = 0, SPMV_JAC0 = 1, SPMV_NOD0 = 2 };

template <class T, int SPL, int LPR, int EP>
__device__ __forceinline__ void spmv_real_row(int64_t t_, int64_t nr, int k, const SellV<T> &M, const C2<T> *__restrict__ x,
                                              C2<T> *__restrict__ y, int accumulate, const T *__restrict__ c1v,
                                              const T *__restrict__ c2v, const Jac0<T> &jz, const Nod0<T> &nz) {
  constexpr int KS = SPL;  // LPR adjacent lanes share a row, SPL slots each
  const int64_t pos = t_ / LPR;
  if (pos >= nr) return;
  const int j0 = ((int)blockIdx.y * LPR + (int)(t_ - pos * LPR)) * SPL;
  const int64_t i = M.rows ? (int64_t)M.rows[pos] : pos;  // slot position -> row
  C2<T> acc[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) acc[q] = {0, 0};
  {
    const int64_t sl = pos >> 6;
    const int lane = (int)(pos & 63);
    const int64_t b0 = M.base[sl];
    const int wd = M.w[sl];
    sell_row<T, KS, 1>(M, b0, wd, lane, x, k, j0, [&](T a, T, T, const C2<T>(&xv)[KS]) {
#pragma unroll
      for (int q = 0; q < KS; ++q) { acc[q].x += a * xv[q].x; acc[q].y += a * xv[q].y; }
    });
  }
  if (EP == SPMV_PLAIN && accumulate) {
    C2<T> o[KS];
    load_slots<T, KS>(y + i * k + j0, o);
#pragma unroll
    for (int q = 0; q < KS; ++q) { acc[q].x += o[q].x; acc[q].y += o[q].y; }
  }
  if (EP != SPMV_NOD0 || y) store_slots<T, KS>(y + i * k + j0, acc);
  if constexpr (EP != SPMV_PLAIN) {
    T c1[KS], c2[KS];
#pragma unroll
    for (int q = 0; q < KS; ++q) { c1[q] = c1v[j0 + q]; c2[q] = c2v[j0 + q]; }
    if constexpr (EP == SPMV_JAC0) {
      jac0_store<T, KS>(jz, i, k, j0, c1, c2, acc);
    } else {
      const T e0 = nz.nd0[i], e1 = nz.nd1[i], m0 = nz.nl0[i], m1 = nz.nl1[i];
      C2<T> o[KS], sm[KS];
      if (nz.sum) load_slots<T, KS>(nz.sum + i * k + j0, sm);
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        const C2<T> dg = l1diag<T>({c1[q] * e0, c2[q] * e1}, fabs(c1[q]) * m0 + c2[q] * m1);
        const C2<T> z = cdiv(acc[q], dg);
        o[q] = {nz.damp * z.x, nz.damp * z.y};
        if (nz.sum) sm[q] = {sm[q].x + o[q].x, sm[q].y + o[q].y};
      }
      store_slots<T, KS>(nz.d + i * k + j0, o);
      if (nz.sum) store_slots<T, KS>(nz.sum + i * k + j0, sm);
    }
  }
}

template <class T, int SPL, int LPR, int EP>
__global__ void __launch_bounds__(256) k_spmv_real_sell(int64_t nr, int k, SellV<T> M, const C2<T> *__restrict__ x,
                                                        C2<T> *__restrict__ y, int accumulate,
                                                        const T *__restrict__ c1v, const T *__restrict__ c2v, Jac0<T> jz,
                                                        Nod0<T> nz) {
  spmv_real_row<T, SPL, LPR, EP>(xcd_block_id() * blockDim.x + threadIdx.x, nr, k, M, x, y, accumulate, c1v, c2v, jz, nz);
}

// y += M x and y2 += M2 x2: workgroups below nb take the first, the others the second
template <class T, int SPL, int LPR>
__global__ void __launch_bounds__(256) k_prolong_sell(unsigned nb, int64_t nr, int64_t nr2, int k, SellV<T> M, SellV<T> M2,
                                                      const C2<T> *__restrict__ x, C2<T> *__restrict__ y,
                                                      const C2<T> *__restrict__ x2, C2<T> *__restrict__ y2) {
  const int64_t b = xcd_block_id();
  if (b < (int64_t)nb)
    spmv_real_row<T, SPL, LPR, SPMV_PLAIN>(b * 256 + threadIdx.x, nr, k, M, x, y, 1, nullptr, nullptr, Jac0<T>(), Nod0<T>());
  else
    spmv_real_row<T, SPL, LPR, SPMV_PLAIN>((b - nb) * 256 + threadIdx.x, nr2, k, M2, x2, y2, 1, nullptr, nullptr, Jac0<T>(),
                                              Nod0<T>());
}

// Products with the auxiliary operators (N, P, P^T, Gx^T): 24 entries or fewer
// in most rows of the finest level, 30-250 in nearly every row of the coarse
// ones, up to 1e5 in the conductor aggregates' rows.  One launch takes all but
// the longest rows whole:
//   * the first nbw workgroups give each chunk of a listed row (kLongRow) a
//     wavefront: LPR lanes hold an entry's SPL slots each, 64 / LPR entries
//     side by side, so the CSR's indices and values are read in order and the
//     walk of 256 entries takes four rounds at 16 slots.  A row of one chunk
//     ends here; the others leave partial sums to k_aux_fin;
//   * the rest walk the short rows' SELL copy, LPR lanes per row.
// Listed and short rows in one SELL copy (the layout before, with separate
// launches for rows above 256 entries) left every launch waiting for its
// longest row: at 48x48x12 with 16 slots 45 / 59 / 65 / 63 us for the residual
// on the four levels, 14 / 9 / 7 / 7 us now, plus 3 us for the rows of several
// chunks.
//   AX_REAL: y (+)= M x, and with z also z = y / d(w)   (the next sweep from 0)
//   AX_RES:  y = r - M(w) x
//   AX_JAC:  y = x + (r - M(w) x) / d(w)
enum AuxMode { AX_REAL = 0, AX_RES = 1, AX_JAC = 2 };

template <class T>
struct AuxEp {
  const C2<T> *r = nullptr;   // AX_RES, AX_JAC
  C2<T> *y = nullptr;
  int accumulate = 0;         // AX_REAL
  C2<T> *z = nullptr;         // AX_REAL
  const T *d0 = nullptr, *d1 = nullptr, *l0 = nullptr, *l1 = nullptr;  // diagonals (of y's level)
};

// what the epilogue of a row reads, loaded before its walk
template <class T, int KS, int MODE>
struct AuxRow {
  C2<T> b[KS], x0[KS];
  T d0, d1, l0, l1;
  __device__ __forceinline__ void load(const AuxEp<T> &ep, const C2<T> *__restrict__ x, int64_t i, int k, int j0) {
    if (MODE != AX_REAL) load_slots<T, KS>(ep.r + i * k + j0, b);
    else if (ep.accumulate) load_slots<T, KS>(ep.y + i * k + j0, b);
    if (MODE == AX_JAC) load_slots<T, KS>(x + i * k + j0, x0);
    if (MODE == AX_JAC || (MODE == AX_REAL && ep.z)) { d0 = ep.d0[i]; d1 = ep.d1[i]; l0 = ep.l0[i]; l1 = ep.l1[i]; }
  }
  __device__ __forceinline__ void store(const AuxEp<T> &ep, int64_t i, int k, int j0, const T (&c1)[KS], const T (&c2)[KS],
                                        const C2<T> (&acc)[KS]) {
    C2<T> o[KS];
#pragma unroll
    for (int q = 0; q < KS; ++q) {
      if (MODE == AX_REAL) o[q] = ep.accumulate ? C2<T>{b[q].x + acc[q].x, b[q].y + acc[q].y} : acc[q];
      else o[q] = {b[q].x - acc[q].x, b[q].y - acc[q].y};
    }
    if (MODE == AX_JAC || (MODE == AX_REAL && ep.z)) {
      C2<T> z[KS];
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        const C2<T> dg = l1diag<T>({c1[q] * d0, c2[q] * d1}, fabs(c1[q]) * l0 + c2[q] * l1);
        z[q] = cdiv(o[q], dg);
        if (MODE == AX_JAC) z[q] = {x0[q].x + z[q].x, x0[q].y + z[q].y};
      }
      if (MODE == AX_JAC) { store_slots<T, KS>(ep.y + i * k + j0, z); return; }
      store_slots<T, KS>(ep.z + i * k + j0, z);
    }
    store_slots<T, KS>(ep.y + i * k + j0, o);
  }
};

template <class T, int SPL, int LPR, int MODE>
__global__ void __launch_bounds__(256) k_aux(int64_t nr, int k, unsigned nbw, SellV<T> S, MatV<T> M,
                                             const T *__restrict__ c1v, const T *__restrict__ c2v,
                                             const C2<T> *__restrict__ x, AuxEp<T> ep, C2<T> *__restrict__ part) {
  constexpr int KS = SPL, G = 64 / LPR;
  C2<T> acc[KS];
  T c1[KS], c2[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) acc[q] = {0, 0};
  AuxRow<T, KS, MODE> row;
  if (blockIdx.x < nbw) {
    const int c = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (c >= M.nchunk) return;  // uniform across the wavefront
    const int lane = threadIdx.x & 63, g = lane / LPR;
    const int j0 = ((int)blockIdx.y * LPR + lane % LPR) * SPL;
#pragma unroll
    for (int q = 0; q < KS; ++q) { c1[q] = c1v[j0 + q]; c2[q] = c2v[j0 + q]; }
    const int64_t b = M.lcb[c], e = M.lce[c];
    const bool whole = c < M.nsingle;
    const int64_t i = whole ? (int64_t)M.lrows[c] : 0;
    if (whole && g == 0) row.load(ep, x, i, k, j0);
    for (int64_t p = b; p < e; p += 4 * G) {
      int32_t ci[4];
      T a0[4], a1[4];
#pragma unroll
      for (int h = 0; h < 4; ++h) {  // past the end: the last entry's column with value 0
        const int64_t t = p + h * G + g;
        const bool in = t < e;
        const int64_t tt = in ? t : e - 1;
        ci[h] = M.ci[tt];
        a0[h] = in ? M.v[0][tt] : (T)0;
        if (MODE != AX_REAL) a1[h] = in ? M.v[1][tt] : (T)0;
      }
      C2<T> xv[4][KS];
#pragma unroll
      for (int h = 0; h < 4; ++h) load_slots<T, KS>(x + (int64_t)ci[h] * k + j0, xv[h]);
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int q = 0; q < KS; ++q) {
          if (MODE == AX_REAL) {
            acc[q].x += a0[h] * xv[h][q].x;
            acc[q].y += a0[h] * xv[h][q].y;
          } else {
            const T ar = c1[q] * a0[h], ai = c2[q] * a1[h];
            acc[q].x += ar * xv[h][q].x - ai * xv[h][q].y;
            acc[q].y += ar * xv[h][q].y + ai * xv[h][q].x;
          }
        }
    }
    es_reduce<T, KS, LPR, G>(acc);
    if (g != 0) return;
    if (whole) row.store(ep, i, k, j0, c1, c2, acc);
    else store_slots<T, KS>(part + (int64_t)(c - M.nsingle) * k + j0, acc);
    return;
  }
  // the short rows: nbw is a multiple of 8, so workgroup b of them sits on
  // XCD b % 8 as xcd_block_id() has it
  const unsigned nb = gridDim.x - nbw, bb = blockIdx.x - nbw;
  const unsigned per = nb >> 3, rem = nb & 7u, xc = bb & 7u;
  const int64_t t_ = (int64_t)(xc * per + (xc < rem ? xc : rem) + (bb >> 3)) * blockDim.x + threadIdx.x;
  const int64_t i = t_ / LPR;
  if (i >= nr || (M.lidx && M.lidx[i] >= 0)) return;
  const int j0 = ((int)blockIdx.y * LPR + (int)(t_ - i * LPR)) * SPL;
#pragma unroll
  for (int q = 0; q < KS; ++q) { c1[q] = c1v[j0 + q]; c2[q] = c2v[j0 + q]; }
  row.load(ep, x, i, k, j0);
  sell_row<T, KS, MODE == AX_REAL ? 1 : 2>(S, S.base[i >> 6], S.w[i >> 6], (int)(i & 63), x, k, j0,
                                           [&](T a0, T a1, T, const C2<T>(&xv)[KS]) {
#pragma unroll
    for (int q = 0; q < KS; ++q) {
      if (MODE == AX_REAL) {
        acc[q].x += a0 * xv[q].x;
        acc[q].y += a0 * xv[q].y;
      } else {
        const T ar = c1[q] * a0, ai = c2[q] * a1;
        acc[q].x += ar * xv[q].x - ai * xv[q].y;
        acc[q].y += ar * xv[q].y + ai * xv[q].x;
      }
    }
  });
  row.store(ep, i, k, j0, c1, c2, acc);
}

// rows of several chunks: one workgroup per row and slot group sums their
// partial sums in a fixed order and ends the row
template <class T, int SPL, int LPR, int MODE>
__global__ void __launch_bounds__(256) k_aux_fin(int k, MatV<T> M, const T *__restrict__ c1v, const T *__restrict__ c2v,
                                                 const C2<T> *__restrict__ x, AuxEp<T> ep,
                                                 const C2<T> *__restrict__ part) {
  constexpr int KS = SPL, G = 64 / LPR;
  __shared__ C2<T> red[4][LPR * KS];
  const int q0 = M.nsingle + (int)blockIdx.x;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, sub = lane % LPR, g = lane / LPR;
  const int j0 = ((int)blockIdx.y * LPR + sub) * SPL;
  C2<T> acc[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) acc[q] = {0, 0};
  for (int c = M.lqp[q0] + wave * G + g; c < M.lqp[q0 + 1]; c += 4 * G) {
    C2<T> v[KS];
    load_slots<T, KS>(part + (int64_t)(c - M.nsingle) * k + j0, v);
#pragma unroll
    for (int q = 0; q < KS; ++q) { acc[q].x += v[q].x; acc[q].y += v[q].y; }
  }
  es_reduce<T, KS, LPR, G>(acc);
  if (g == 0)
#pragma unroll
    for (int q = 0; q < KS; ++q) red[wave][sub * KS + q] = acc[q];
  __syncthreads();
  if (threadIdx.x >= LPR) return;
  T c1[KS], c2[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) {
    c1[q] = c1v[j0 + q];
    c2[q] = c2v[j0 + q];
    for (int w = 1; w < 4; ++w) { acc[q].x += red[w][sub * KS + q].x; acc[q].y += red[w][sub * KS + q].y; }
  }
  AuxRow<T, KS, MODE> row;
  const int64_t i = M.lrows[q0];
  row.load(ep, x, i, k, j0);
  row.store(ep, i, k, j0, c1, c2, acc);
}

// SELL y -= M2(w) x, M2 = c1 v0 + i c2 v1
template <class T, int SPL, int LPR>
__global__ void __launch_bounds__(256) k_spmv2_sell(int64_t nr, int k, SellV<T> M, const T *__restrict__ c1v,
                                                    const T *__restrict__ c2v, const C2<T> *__restrict__ x,
                                                    C2<T> *__restrict__ y, Jac0<T> jz) {
  constexpr int KS = SPL;  // LPR adjacent lanes share a row, SPL slots each
  const int64_t t_ = xcd_block_id() * blockDim.x + threadIdx.x;
  const int64_t pos = t_ / LPR;
  if (pos >= nr) return;
  const int j0 = ((int)blockIdx.y * LPR + (int)(t_ - pos * LPR)) * SPL;
  const int64_t i = M.rows ? (int64_t)M.rows[pos] : pos;  // slot position -> row
  T c1[KS], c2[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) { c1[q] = c1v[j0 + q]; c2[q] = c2v[j0 + q]; }
  C2<T> acc[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) acc[q] = {0, 0};
  {
    const int64_t sl = pos >> 6;
    const int lane = (int)(pos & 63);
    const int64_t b0 = M.base[sl];
    const int wd = M.w[sl];
    sell_row<T, KS, 2>(M, b0, wd, lane, x, k, j0, [&](T a0, T a1, T, const C2<T>(&xv)[KS]) {
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        const T ar = c1[q] * a0, ai = c2[q] * a1;
        acc[q].x += ar * xv[q].x - ai * xv[q].y;
        acc[q].y += ar * xv[q].y + ai * xv[q].x;
      }
    });
  }
  C2<T> o[KS];
  load_slots<T, KS>(y + i * k + j0, o);
#pragma unroll
  for (int q = 0; q < KS; ++q) o[q] = {o[q].x - acc[q].x, o[q].y - acc[q].y};
  store_slots<T, KS>(y + i * k + j0, o);
  if (jz.u) jac0_store<T, KS>(jz, i, k, j0, c1, c2, o);
}

// k_spmv2_sell on an operator of kNok2MinRows rows or more (the level-0 Bx
// product): two rows per lane group, their indices and values, y and the
// epilogue's diagonals
// loaded before the row gathers, as in k_edge_nok2.  Per row the entries are
// summed in the same order; the compiler may fuse the complex products'
// multiply-adds differently from k_spmv2_sell (Z of a 400x400x32 solve moved
// by 5e-15 relative, same iterations).
template <class T, int SPL, int LPR>
__global__ void __launch_bounds__(256) k_spmv2_sell2(int64_t nr, int64_t half, int k, SellV<T> M,
                                                     const T *__restrict__ c1v, const T *__restrict__ c2v,
                                                     const C2<T> *__restrict__ x, C2<T> *__restrict__ y,
                                                     Jac0<T> jz) {
  constexpr int KS = SPL, NR = 2, PF = 4;
  const int64_t t = xcd_block_id() * blockDim.x + threadIdx.x;
  const int64_t q0 = t / LPR;
  if (q0 >= half) return;
  const int j0 = ((int)blockIdx.y * LPR + (int)(t - q0 * LPR)) * SPL;
  T c1[KS], c2[KS];
#pragma unroll
  for (int q = 0; q < KS; ++q) { c1[q] = c1v[j0 + q]; c2[q] = c2v[j0 + q]; }
  bool ok[NR];
  int64_t i[NR], b0[NR];
  int wd[NR], lane[NR];
  int32_t c[NR][PF];
  T a0[NR][PF], a1[NR][PF];
  C2<T> o[NR][KS], acc[NR][KS];
  T d[NR][6];
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    const int64_t pos = q0 + n * half;
    ok[n] = pos < nr;
    i[n] = 0; b0[n] = 0; wd[n] = 0; lane[n] = 0;
#pragma unroll
    for (int q = 0; q < KS; ++q) acc[n][q] = {0, 0};
    if (!ok[n]) continue;
    i[n] = M.rows ? (int64_t)M.rows[pos] : pos;
    const int64_t sl = pos >> 6;
    lane[n] = (int)(pos & 63);
    b0[n] = M.base[sl];
    wd[n] = M.w[sl];
  }
#pragma unroll
  for (int n = 0; n < NR; ++n) {
#pragma unroll
    for (int h = 0; h < PF; ++h) {
      c[n][h] = 0; a0[n][h] = (T)0; a1[n][h] = (T)0;
      if (h < wd[n]) {
        const int64_t e = b0[n] + (int64_t)h * 64 + lane[n];
        c[n][h] = __builtin_nontemporal_load(M.ci + e);
        a0[n][h] = __builtin_nontemporal_load(M.v[0] + e);
        a1[n][h] = __builtin_nontemporal_load(M.v[1] + e);
      }
    }
    if (!ok[n]) continue;
    load_slots<T, KS>(y + i[n] * k + j0, o[n]);
    if (jz.u) {
      d[n][0] = jz.kd0[i[n]]; d[n][1] = jz.kd1[i[n]]; d[n][2] = jz.kd2[i[n]];
      d[n][3] = jz.kl0[i[n]]; d[n][4] = jz.kl1[i[n]]; d[n][5] = jz.kl2[i[n]];
    }
  }
#pragma unroll
  for (int t0 = 0; t0 < PF; t0 += 2) {  // two gathers per row in flight
    C2<T> xv[NR][2][KS];
#pragma unroll
    for (int n = 0; n < NR; ++n)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (t0 + h < wd[n]) load_slots<T, KS>(x + (int64_t)c[n][t0 + h] * k + j0, xv[n][h]);
#pragma unroll
    for (int n = 0; n < NR; ++n)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (t0 + h < wd[n])
#pragma unroll
          for (int q = 0; q < KS; ++q) {
            const T ar = c1[q] * a0[n][t0 + h], ai = c2[q] * a1[n][t0 + h];
            acc[n][q].x += ar * xv[n][h][q].x - ai * xv[n][h][q].y;
            acc[n][q].y += ar * xv[n][h][q].y + ai * xv[n][h][q].x;
          }
  }
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    if (!ok[n]) continue;
    auto f = [&](T b0v, T b1v, T, const C2<T>(&xr)[KS]) {
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        const T ar = c1[q] * b0v, ai = c2[q] * b1v;
        acc[n][q].x += ar * xr[q].x - ai * xr[q].y;
        acc[n][q].y += ar * xr[q].y + ai * xr[q].x;
      }
    };
    for (int tt = PF; tt < wd[n]; ++tt) sell_batch<T, KS, 2, 1, 1>(M, b0[n], tt, lane[n], x, k, j0, f);
#pragma unroll
    for (int q = 0; q < KS; ++q) o[n][q] = {o[n][q].x - acc[n][q].x, o[n][q].y - acc[n][q].y};
    store_slots<T, KS>(y + i[n] * k + j0, o[n]);
    if (jz.u) {
      C2<T> uo[KS];
#pragma unroll
      for (int q = 0; q < KS; ++q) {
        const C2<T> dq = l1diag<T>({d[n][0] + c1[q] * d[n][1], c2[q] * d[n][2]},
                                   d[n][3] + fabs(c1[q]) * d[n][4] + c2[q] * d[n][5]);
        const C2<T> z = cdiv(o[n][q], dq);
        uo[q] = {jz.damp * z.x, jz.damp * z.y};
      }
      store_slots<T, KS>(jz.u + i[n] * k + j0, uo);
    }
  }
}

// Nodal l1-Jacobi on N(w) = -w^2 N_eps + i w N_sig:
//   first (d == null): d_out = rn / dn;  else d_out = d + (rn - N d) / dn
template <class T>
__global__ void k_node(int64_t nr, int k, MatV<T> N, const T *__restrict__ c1v, const T *__restrict__ c2v,
                       const T *__restrict__ nd0, const T *__restrict__ nd1, const T *__restrict__ nl0,
                       const T *__restrict__ nl1, const C2<T> *__restrict__ rn, const C2<T> *__restrict__ d,
                       C2<T> *__restrict__ dout, T damp, const C2<T> *__restrict__ lp) {
  int64_t t = xcd_block_id() * blockDim.x + threadIdx.x;
  int64_t i = t / k;
  int j = (int)(t - i * k);
  if (i >= nr) return;
  const T c1 = c1v[j], c2 = c2v[j];
  C2<T> acc = rn[i * k + j];
  const int32_t q = (d && N.lidx) ? N.lidx[i] : -1;
  if (q >= 0) {
    const C2<T> s0 = lp[((int64_t)q * 2) * k + j], s1 = lp[((int64_t)q * 2 + 1) * k + j];
    acc.x -= c1 * s0.x - c2 * s1.y;
    acc.y -= c1 * s0.y + c2 * s1.x;
  } else if (d) {
    for (int64_t p = N.rp[i]; p < N.rp[i + 1]; ++p) {
      C2<T> a = {c1 * N.v[0][p], c2 * N.v[1][p]};
      C2<T> x = d[(int64_t)N.ci[p] * k + j];
      acc.x -= a.x * x.x - a.y * x.y;
      acc.y -= a.x * x.y + a.y * x.x;
    }
  }
  C2<T> dg = l1diag<T>({c1 * nd0[i], c2 * nd1[i]}, fabs(c1) * nl0[i] + c2 * nl1[i]);
  C2<T> dq = cdiv(acc, dg);
  if (!d) { dout[i * k + j] = {damp * dq.x, damp * dq.y}; return; }
  C2<T> d0 = d[i * k + j];
  dout[i * k + j] = {d0.x + damp * dq.x, d0.y + damp * dq.y};
}

// y = M x (real matrix, complex multi-column vectors); accumulate adds to y.
template <class T>
__global__ void k_spmv_real(int64_t nr, int k, MatV<T> M, const C2<T> *__restrict__ x, C2<T> *__restrict__ y, int accumulate,
                            const C2<T> *__restrict__ lp) {
  int64_t t = xcd_block_id() * blockDim.x + threadIdx.x;
  int64_t i = t / k;
  int j = (int)(t - i * k);
  if (i >= nr) return;
  C2<T> acc = {0, 0};
  const int32_t q = M.lidx ? M.lidx[i] : -1;
  if (q >= 0) acc = lp[(int64_t)q * k + j];
  else for (int64_t p = M.rp[i]; p < M.rp[i + 1]; ++p) {
    const T a = M.v[0][p];
    C2<T> v = x[(int64_t)M.ci[p] * k + j];
    acc.x += a * v.x;
    acc.y += a * v.y;
  }
  if (accumulate) { C2<T> o = y[i * k + j]; acc.x += o.x; acc.y += o.y; }
  y[i * k + j] = acc;
}

template <class T>
__global__ void k_add(int64_t n, C2<T> *__restrict__ a, const C2<T> *__restrict__ b) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) { a[i].x += b[i].x; a[i].y += b[i].y; }
}

// Exact coarsest solve in FP64 of k columns,
//   phi = N^-1 (G^T r);  rs = r - B phi;  u = K^-1 rs,
// as three dense products, each spread over the chip with a wavefront per
// row: N^-1 G^T is kept per frequency (coarse_cache_lookup).  The level has at
// most ~400 edges, so the products are bound by latency and, where one
// workgroup walks a column's matrices alone, by what one CU can load: one
// workgroup per column with a thread per row, each lane reading its own line
// per entry, took 213 us at 48x48x12 (266 edges, 98 nodes, 16 columns); with
// 16 lanes per row in one workgroup 23 us plus 4 for u; these take 16 us.
template <class T, class TX>
__device__ __forceinline__ C2<double> dense_row(int64_t nc, const C2<double> *__restrict__ M,
                                                const C2<TX> *__restrict__ x, int64_t xs) {
  const int lane = threadIdx.x & 63;
  C2<double> t = {0., 0.};
#pragma unroll 4
  for (int64_t b = lane; b < nc; b += 64) {
    const C2<double> m = M[b];
    const C2<TX> v = x[b * xs];
    t.x += m.x * (double)v.x - m.y * (double)v.y;
    t.y += m.x * (double)v.y + m.y * (double)v.x;
  }
  for (int o = 32; o > 0; o >>= 1) { t.x += __shfl_xor(t.x, o); t.y += __shfl_xor(t.y, o); }
  return t;
}

// step 0: phi (T and, column by column, FP64 in ph); 1: rs; 2: u.  Grid
// (rows / 4, columns).
template <class T>
__global__ void __launch_bounds__(256) k_coarse(int step, int64_t ne, int64_t nn, int k, const int32_t *__restrict__ fidx,
                                                const double *const *__restrict__ tab, int cap,
                                                const C2<T> *__restrict__ r, C2<double> *__restrict__ ph,
                                                C2<double> *__restrict__ rs, C2<T> *__restrict__ phi,
                                                C2<T> *__restrict__ u) {
  const int j = blockIdx.y;
  const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= (step == 0 ? nn : ne)) return;  // uniform across the wavefront
  const int f = fidx[j];
  const bool first = (threadIdx.x & 63) == 0;
  if (step == 0) {
    const C2<double> t = dense_row<T, T>(ne, (const C2<double> *)tab[cap + f] + i * ne, r + j, k);
    if (first) { ph[(int64_t)j * nn + i] = t; phi[i * k + j] = {(T)t.x, (T)t.y}; }
  } else if (step == 1) {
    const C2<T> r0 = r[i * k + j];
    const C2<double> t = dense_row<T, double>(nn, (const C2<double> *)tab[2 * cap + f] + i * nn, ph + (int64_t)j * nn, 1);
    if (first) rs[(int64_t)j * ne + i] = {(double)r0.x - t.x, (double)r0.y - t.y};
  } else {
    const C2<double> t = dense_row<T, double>(ne, (const C2<double> *)tab[f] + i * ne, rs + (int64_t)j * ne, 1);
    if (first) u[i * k + j] = {(T)t.x, (T)t.y};
  }
}

// y = r - M2(w) x, M2 = c1 v0 + i c2 v1 (r may be y)
template <class T>
__global__ void k_spmv2(int64_t nr, int k, MatV<T> M, const T *__restrict__ c1v, const T *__restrict__ c2v,
                        const C2<T> *r, const C2<T> *__restrict__ x, C2<T> *y, const C2<T> *__restrict__ lp) {
  int64_t t = xcd_block_id() * blockDim.x + threadIdx.x;
  int64_t i = t / k;
  int j = (int)(t - i * k);
  if (i >= nr) return;
  const T c1 = c1v[j], c2 = c2v[j];
  C2<T> acc = {0, 0};
  const int32_t q = M.lidx ? M.lidx[i] : -1;
  if (q >= 0) {
    const C2<T> s0 = lp[((int64_t)q * 2) * k + j], s1 = lp[((int64_t)q * 2 + 1) * k + j];
    acc = {c1 * s0.x - c2 * s1.y, c1 * s0.y + c2 * s1.x};
  } else for (int64_t p = M.rp[i]; p < M.rp[i + 1]; ++p) {
    C2<T> a = {c1 * M.v[0][p], c2 * M.v[1][p]};
    C2<T> v = x[(int64_t)M.ci[p] * k + j];
    acc.x += a.x * v.x - a.y * v.y;
    acc.y += a.x * v.y + a.y * v.x;
  }
  const C2<T> b = r[i * k + j];
  y[i * k + j] = {b.x - acc.x, b.y - acc.y};
}

// x = A_f^-1 r at the auxiliary coarsest level, A_f block diagonal
// (AuxAMG::nblk) with the block inverses packed per frequency: position i
// (coarse index perm[i]) of block B sums over B's columns only.  Grid
// (positions / 4, columns): one wavefront per position, products in FP64.
template <class T>
__global__ void __launch_bounds__(256) k_blkdiag_apply(int64_t n, int k, const int32_t *__restrict__ perm,
                                                       const int32_t *__restrict__ rowblk,
                                                       const int32_t *__restrict__ boff,
                                                       const int64_t *__restrict__ ioff,
                                                       const int32_t *__restrict__ fidx,
                                                       const double *const *__restrict__ tab,
                                                       const C2<T> *__restrict__ r, C2<T> *__restrict__ x) {
  const int j = blockIdx.y;
  const C2<double> *M = (const C2<double> *)tab[fidx[j]];
  const int lane = threadIdx.x & 63;
  const int64_t i = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (i >= n) return;
  const int B = rowblk[i];
  const int o = boff[B], b = boff[B + 1] - o;
  const C2<double> *R = M + ioff[B] + (int64_t)(i - o) * b;
  double ax = 0, ay = 0;
  for (int c = lane; c < b; c += 64) {
    const C2<double> m = R[c];
    const C2<T> v = r[(int64_t)perm[o + c] * k + j];
    ax += m.x * (double)v.x - m.y * (double)v.y;
    ay += m.x * (double)v.y + m.y * (double)v.x;
  }
  for (int off = 32; off > 0; off >>= 1) {
    ax += __shfl_xor(ax, off);
    ay += __shfl_xor(ay, off);
  }
  if (lane == 0) x[(int64_t)perm[i] * k + j] = {(T)ax, (T)ay};
}

template <class T>
__global__ void k_copy(int64_t n, const C2<T> *__restrict__ a, C2<T> *__restrict__ b) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

template <class T>
MatV<T> view(const Csr &c, const CsrF &f);
template <>
MatV<double> view<double>(const Csr &c, const CsrF &) {
  MatV<double> v; v.nr = c.nr; v.nc = c.nc; v.rp = c.rp; v.ci = c.ci; v.nv = c.nv;
  for (int k = 0; k < c.nv; ++k) v.v[k] = c.v[k];
  v.nlong = c.nlong; v.lrows = c.lrows; v.lidx = c.lidx;
  v.nchunk = c.nchunk; v.nsingle = c.nsingle; v.lcb = c.lcb; v.lce = c.lce; v.lqp = c.lqp;
  v.dg[0] = c.dg[0]; v.dg[1] = c.dg[1];
  return v;
}
template <>
MatV<float> view<float>(const Csr &, const CsrF &f) {
  MatV<float> v; v.nr = f.nr; v.nc = f.nc; v.rp = f.rp; v.ci = f.ci; v.nv = f.nv;
  for (int k = 0; k < f.nv; ++k) v.v[k] = f.v[k];
  v.nlong = f.nlong; v.lrows = f.lrows; v.lidx = f.lidx;
  v.nchunk = f.nchunk; v.nsingle = f.nsingle; v.lcb = f.lcb; v.lce = f.lce; v.lqp = f.lqp;
  v.dg[0] = f.dg[0]; v.dg[1] = f.dg[1];
  return v;
}

template <class T>
SellV<T> sview(const Sell &c, const SellF &f, const Csr &kc, const CsrF &kf);
template <>
SellV<double> sview<double>(const Sell &c, const SellF &, const Csr &kc, const CsrF &) {
  SellV<double> v; v.nr = c.nr; v.nslice = c.nslice; v.nent = c.nent; v.base = c.base; v.w = c.w; v.ci = c.ci; v.nv = c.nv;
  for (int q = 0; q < c.nv; ++q) v.v[q] = c.v[q];
  v.dg[0] = kc.dg[0]; v.dg[1] = kc.dg[1]; v.dgs = kc.sdg;
  v.rows = c.rows;
  return v;
}
template <>
SellV<float> sview<float>(const Sell &, const SellF &f, const Csr &, const CsrF &kf) {
  SellV<float> v; v.nr = f.nr; v.nslice = f.nslice; v.nent = f.nent; v.base = f.base; v.w = f.w; v.ci = f.ci; v.nv = f.nv;
  for (int q = 0; q < f.nv; ++q) v.v[q] = f.v[q];
  v.dg[0] = kf.dg[0]; v.dg[1] = kf.dg[1]; v.dgs = kf.sdg;
  v.rows = f.rows;
  return v;
}

// Kernel choice per operator: the lanes-per-row SELL kernels for operators of
// at least sell_min_rows rows (default 1: every operator), else the (row,
// slot) CSR kernels.  Measured at 200x200x24, 80 columns, with four gathers
// in flight per lane: 15.1 solves/s with SELL everywhere, 15.0 from 4096
// rows, 14.7 from 2^14, 14.2 from 2^16.
// Launch shape of the lanes-per-row SELL kernels: SPL slots per lane (FP32:
// 4 when k allows -- two 16-byte loads per gathered row --, else 2 or 1;
// FP64: 1), LPR lanes per row (the largest power of two up to 16 that divides
// k / SPL), k / (SPL LPR) grid rows.  Measured at 200x200x24, 16 slots, level-0
// edge smoother: SPL 2 / LPR 8 536 us, SPL 4 / LPR 4 499 us, SPL 8 / LPR 2
// 534 us (and the whole solve 27 % slower: register pressure).
struct Lanes {
  int sp = 1, lpr = 1;
  dim3 grid;
};
thread_local int t_lanes_cap = 16;

template <class T>
Lanes lanes_shape(int64_t nr, int k) {
  Lanes L;
  if (sizeof(T) == 4) L.sp = (k % 4 == 0) ? 4 : (k % 2 == 0) ? 2 : 1;
  while (L.lpr < t_lanes_cap && (k / L.sp) % (L.lpr * 2) == 0) L.lpr *= 2;
  L.grid = dim3((unsigned)((nr * L.lpr + 255) / 256), (unsigned)(k / (L.sp * L.lpr)));
  return L;
}

// go(slots per lane, lanes per row) as compile-time constants
template <class T, class F>
void lanes_go(const Lanes &ln, F &&go) {
  auto lanes = [&](auto sp_) {
    if (ln.lpr == 16) go(sp_, std::integral_constant<int, 16>());
    else if (ln.lpr == 8) go(sp_, std::integral_constant<int, 8>());
    else if (ln.lpr == 4) go(sp_, std::integral_constant<int, 4>());
    else if (ln.lpr == 2) go(sp_, std::integral_constant<int, 2>());
    else go(sp_, std::integral_constant<int, 1>());
  };
  if constexpr (sizeof(T) == 4) {
    if (ln.sp == 4) { lanes(std::integral_constant<int, 4>()); return; }
    if (ln.sp == 2) { lanes(std::integral_constant<int, 2>()); return; }
  }
  lanes(std::integral_constant<int, 1>());
}

// Entry groups per row of the nodal sweep with one slot (the plain FP64
// single-column path), from the operator's stored entries per row (slice widths,
// padding included): a single lane walks the 27 entries of a coarse level's row
// serially.  With more slots a row has more lanes, and the launches are bound by
// the slot data that each entry gathers, not by the walk.  The other operators
// here hold at most 18 entries a row (coarse edges restrict 2 x 3 x 3 fine ones).
template <class T>
int entry_split(const SellV<T> &M, const Lanes &L) {
  if (!(L.sp == 1 && L.lpr == 1) || M.nr == 0) return 1;
  return (double)M.nent / (double)M.nr >= 24 ? 4 : 1;
}

template <class T>
void edge_sell(int64_t nr, int64_t smin, int k, const SellV<T> &K, const SellV<T> &B, const MatV<T> &Kc, const MatV<T> &Bc,
               const T *c1, const T *c2, const T *kd0, const T *kd1, const T *kd2, const T *kl0, const T *kl1,
               const T *kl2, const C2<T> *r, const C2<T> *u, const C2<T> *phi, C2<T> *out, int mode, int use_phi,
               T damp, hipStream_t s) {
  if (nr < smin) {
    k_edge<T><<<blocks_for(nr * k), 256, 0, s>>>(nr, k, Kc, Bc, c1, c2, kd0, kd1, kd2, kl0, kl1, kl2, r, u, phi, out,
                                                 mode, use_phi, damp);
    return;
  }
  const int kind = mode & EdgeMode::KIND;
  // no K u on an operator whose vectors stream from HBM: two rows per lane
  // group.  At 400x400x32 the level-0 launches (15.4M rows) took 1252 us
  // against 2010 us; on level 1 (1.9M rows, its vectors held in the caches)
  // the single-row kernel is faster (276 us against 374 us)
  if (((mode & EdgeMode::NOK) || kind == EdgeMode::JACOBI0) && nr >= kNok2MinRows) {
    const int64_t half = (nr + 1) / 2;
    const Lanes ln = lanes_shape<T>(half, k);
    if (ln.sp == 4) {
#define GP_NOK2(L) k_edge_nok2<T, 4, L><<<ln.grid, 256, 0, s>>>(nr, half, k, K, B, c1, c2, kd0, kd1, kd2, kl0, kl1, kl2, \
                                                                r, u, phi, out, mode, use_phi, damp)
      if (ln.lpr == 16) GP_NOK2(16);
      else if (ln.lpr == 8) GP_NOK2(8);
      else if (ln.lpr == 4) GP_NOK2(4);
      else if (ln.lpr == 2) GP_NOK2(2);
      else GP_NOK2(1);
#undef GP_NOK2
      return;
    }
  }
  const Lanes ln = lanes_shape<T>(nr, k);
  lanes_go<T>(ln, [&](auto sp_, auto lp_) {
    k_edge_sell<T, decltype(sp_)::value, decltype(lp_)::value>
        <<<ln.grid, 256, 0, s>>>(nr, k, K, B, c1, c2, kd0, kd1, kd2, kl0, kl1, kl2, r, u, phi, out, mode, use_phi, damp);
  });
}

template <class T>
SellV<T> sv(const Sell &c, const SellF &f);
template <>
SellV<double> sv<double>(const Sell &c, const SellF &) {
  SellV<double> v; v.nr = c.nr; v.nslice = c.nslice; v.nent = c.nent; v.base = c.base; v.w = c.w; v.ci = c.ci; v.nv = c.nv;
  for (int q = 0; q < c.nv; ++q) v.v[q] = c.v[q];
  v.rows = c.rows;
  return v;
}
template <>
SellV<float> sv<float>(const Sell &, const SellF &f) {
  SellV<float> v; v.nr = f.nr; v.nslice = f.nslice; v.nent = f.nent; v.base = f.base; v.w = f.w; v.ci = f.ci; v.nv = f.nv;
  for (int q = 0; q < f.nv; ++q) v.v[q] = f.v[q];
  v.rows = f.rows;
  return v;
}

template <class T>
void node_sell(int64_t nr, int64_t smin, int k, const SellV<T> &N, const MatV<T> &Nc, const T *c1, const T *c2, const T *nd0,
               const T *nd1, const T *nl0, const T *nl1, const C2<T> *rn, const C2<T> *d, C2<T> *dout, T damp,
               hipStream_t s) {
  if (nr == 0) return;
  if (nr < smin) {
    k_node<T><<<blocks_for(nr * k), 256, 0, s>>>(nr, k, Nc, c1, c2, nd0, nd1, nl0, nl1, rn, d, dout, damp, nullptr);
    return;
  }
  const Lanes ln = lanes_shape<T>(nr, k);
  if (entry_split<T>(N, ln) == 4) {
    k_node_sell<T, 1, 1, 4><<<dim3((unsigned)((nr * 4 + 255) / 256), ln.grid.y), 256, 0, s>>>(
        nr, k, N, c1, c2, nd0, nd1, nl0, nl1, rn, d, dout, damp);
    return;
  }
  lanes_go<T>(ln, [&](auto sp_, auto lp_) {
    k_node_sell<T, decltype(sp_)::value, decltype(lp_)::value, 1>
        <<<ln.grid, 256, 0, s>>>(nr, k, N, c1, c2, nd0, nd1, nl0, nl1, rn, d, dout, damp);
  });
}

template <class T, int EP = SPMV_PLAIN>
void spmv_real_sell(int64_t nr, int64_t smin, int k, const SellV<T> &M, const MatV<T> &Mc, const C2<T> *x, C2<T> *y, int accumulate,
                    hipStream_t s, const T *c1 = nullptr, const T *c2 = nullptr, const Jac0<T> &jz = Jac0<T>(),
                    const Nod0<T> &nz = Nod0<T>()) {
  if (nr == 0) return;
  if (nr < smin) {
    k_spmv_real<T><<<blocks_for(nr * k), 256, 0, s>>>(nr, k, Mc, x, y, accumulate, nullptr);
    return;
  }
  const Lanes ln = lanes_shape<T>(nr, k);
  lanes_go<T>(ln, [&](auto sp_, auto lp_) {
    k_spmv_real_sell<T, decltype(sp_)::value, decltype(lp_)::value, EP>
        <<<ln.grid, 256, 0, s>>>(nr, k, M, x, y, accumulate, c1, c2, jz, nz);
  });
}

// y += M x and y2 += M2 x2 in one launch
template <class T>
void prolong_sell(int64_t nr, int64_t nr2, int64_t smin, int k, const SellV<T> &M, const MatV<T> &Mc, const C2<T> *x, C2<T> *y,
                  const SellV<T> &M2, const MatV<T> &M2c, const C2<T> *x2, C2<T> *y2, hipStream_t s) {
  const Lanes ln = lanes_shape<T>(nr, k), l2 = lanes_shape<T>(nr2, k);
  if (nr == 0 || nr2 == 0 || nr < smin || nr2 < smin) {
    spmv_real_sell<T>(nr, smin, k, M, Mc, x, y, 1, s);
    spmv_real_sell<T>(nr2, smin, k, M2, M2c, x2, y2, 1, s);
    return;
  }
  const dim3 grid(ln.grid.x + l2.grid.x, ln.grid.y);
  const unsigned nb = ln.grid.x;
  auto go = [&](auto sp_, auto lp_) {
    k_prolong_sell<T, decltype(sp_)::value, decltype(lp_)::value>
        <<<grid, 256, 0, s>>>(nb, nr, nr2, k, M, M2, x, y, x2, y2);
  };
  lanes_go<T>(ln, go);
}

// y -= M2(w) x.  Returns whether the optional epilogue jz ran (sliced-ELL path only).
template <class T>
bool spmv2_sell(int64_t nr, int64_t smin, int k, const SellV<T> &M, const MatV<T> &Mc, const T *c1, const T *c2,
                const C2<T> *x, C2<T> *y, hipStream_t s, const Jac0<T> &jz = Jac0<T>()) {
  if (nr == 0) return false;
  if (nr < smin) {
    k_spmv2<T><<<blocks_for(nr * k), 256, 0, s>>>(nr, k, Mc, c1, c2, y, x, y, nullptr);
    return false;
  }
  if (nr >= kNok2MinRows) {  // large operator: two rows per lane group
    const int64_t half = (nr + 1) / 2;
    const Lanes ln = lanes_shape<T>(half, k);
    if (ln.sp == 4) {
#define GP_SPMV2X(L) k_spmv2_sell2<T, 4, L><<<ln.grid, 256, 0, s>>>(nr, half, k, M, c1, c2, x, y, jz)
      if (ln.lpr == 16) GP_SPMV2X(16);
      else if (ln.lpr == 8) GP_SPMV2X(8);
      else if (ln.lpr == 4) GP_SPMV2X(4);
      else if (ln.lpr == 2) GP_SPMV2X(2);
      else GP_SPMV2X(1);
#undef GP_SPMV2X
      return jz.u != nullptr;
    }
  }
  const Lanes ln = lanes_shape<T>(nr, k);
  lanes_go<T>(ln, [&](auto sp_, auto lp_) {
    k_spmv2_sell<T, decltype(sp_)::value, decltype(lp_)::value><<<ln.grid, 256, 0, s>>>(nr, k, M, c1, c2, x, y, jz);
  });
  return jz.u != nullptr;
}

template <class T> const T *arr(double *d, float *f);
template <> const double *arr<double>(double *d, float *) { return d; }
template <> const float *arr<float>(double *, float *f) { return f; }

inline unsigned grid_rows(int64_t nr, int k) { return blocks_for(nr * k); }

template <class T>
void long_pass(const MatV<T> &M, int k, const C2<T> *x, C2<T> *part, C2<T> *lp, hipStream_t s) {
  if (M.nlong <= 0) return;
  k_long_part<T><<<M.nchunk, 256, 0, s>>>(M, k, x, part);
  k_long_fin<T><<<M.nlong, 256, 0, s>>>(M, k, part, lp);
}

template <class T, int MODE>
void aux_prod(int64_t nr, const VWork<T> &w, const SellV<T> &S, const MatV<T> &M, const C2<T> *x, const AuxEp<T> &ep,
              hipStream_t s) {
  if (nr == 0) return;
  const int k = w.k;
  if (nr < w.sell_min_rows) {
    long_pass<T>(M, k, x, w.lpart, w.lp, s);
    const unsigned g = blocks_for(nr * k);
    if (MODE == AX_JAC)
      k_node<T><<<g, 256, 0, s>>>(nr, k, M, w.c1, w.c2, ep.d0, ep.d1, ep.l0, ep.l1, ep.r, x, ep.y, (T)1, w.lp);
    else if (MODE == AX_RES)
      k_spmv2<T><<<g, 256, 0, s>>>(nr, k, M, w.c1, w.c2, ep.r, x, ep.y, w.lp);
    else
      k_spmv_real<T><<<g, 256, 0, s>>>(nr, k, M, x, ep.y, ep.accumulate, w.lp);
    if (MODE == AX_REAL && ep.z)
      k_node<T><<<g, 256, 0, s>>>(nr, k, M, w.c1, w.c2, ep.d0, ep.d1, ep.l0, ep.l1, ep.y, nullptr, ep.z, (T)1, nullptr);
    return;
  }
  const Lanes ln = lanes_shape<T>(nr, k);
  const unsigned nbw = (unsigned)(((M.nchunk + 3) / 4 + 7) / 8 * 8);
  const unsigned nbs = M.nlong == nr ? 0u : ln.grid.x;
  const dim3 grid(nbw + nbs, ln.grid.y);
  const unsigned nfin = (unsigned)(M.nlong - M.nsingle);
  auto go = [&](auto sp_, auto lp_) {
    constexpr int SP = decltype(sp_)::value, LP = decltype(lp_)::value;
    k_aux<T, SP, LP, MODE><<<grid, 256, 0, s>>>(nr, k, nbw, S, M, w.c1, w.c2, x, ep, w.lpart);
    if (nfin) k_aux_fin<T, SP, LP, MODE><<<dim3(nfin, grid.y), 256, 0, s>>>(k, M, w.c1, w.c2, x, ep, w.lpart);
  };
  lanes_go<T>(ln, go);
}

}  // namespace

// LDS a march workgroup may take on the current device (0: none), with the
// kernels' dynamic-LDS limit raised to it; called while the hierarchy is
// built, outside any stream capture
int march_lds_setup() {
  int d = 0, v = 0;
  if (hipGetDevice(&d) != hipSuccess || hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, d) != hipSuccess)
    return 0;
  if (hipFuncSetAttribute((const void *)k_edge_march<4>, hipFuncAttributeMaxDynamicSharedMemorySize, v) != hipSuccess ||
      hipFuncSetAttribute((const void *)k_edge_march<2>, hipFuncAttributeMaxDynamicSharedMemorySize, v) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return v;
}


// First edge sweep of level l, into the buffer that vcycle_level starts from
template <class T>
static Jac0<T> jac0_of(const MgLevel &L, const VWork<T> &w, int l, int nu_pre, int nu_post) {
  Jac0<T> jz;
  jz.kd0 = arr<T>(L.kd[0], L.kdf[0]); jz.kd1 = arr<T>(L.kd[1], L.kdf[1]); jz.kd2 = arr<T>(L.kd[2], L.kdf[2]);
  jz.kl0 = arr<T>(L.kl[0], L.klf[0]); jz.kl1 = arr<T>(L.kl[1], L.klf[1]); jz.kl2 = arr<T>(L.kl[2], L.klf[2]);
  jz.u = (((nu_pre - 1) + nu_post) & 1) ? w.tmp[l] : w.u[l];
  return jz;
}

template <class T>
static gp_status vcycle_level(const Hierarchy &H, VWork<T> &w, hipStream_t s, int l, int nu_pre, int nu_post) {
  const MgLevel &L = H.L[l];
  const int k = w.k;
  const int64_t ne = L.ne, nn = L.nn;
  C2<T> *r = w.r[l], *u = w.u[l], *phi = w.phi[l], *res = w.res[l], *tmp = w.tmp[l];
  C2<T> *rn = w.rn[l], *d1 = w.dn[l], *d2 = w.dn2[l];
  if (l + 1 == (int)H.L.size()) {
    C2<double> *ph = w.crs, *rs = w.crs + nn * k;
    for (int step = 0; step < 3; ++step) {
      const dim3 grid((unsigned)(((step == 0 ? nn : ne) + 3) / 4), (unsigned)k);
      if (grid.x) k_coarse<T><<<grid, 256, 0, s>>>(step, ne, nn, k, w.fidx, w.tab, w.cap, r, ph, rs, phi, u);
    }
    return GP_OK;
  }
  const MatV<T> K = view<T>(L.K, L.Kf), B = view<T>(L.B, L.Bf), N = view<T>(L.N, L.Nf);
  const SellV<T> KS = sview<T>(L.Ks, L.Ksf, L.K, L.Kf), BS = sview<T>(L.Bs, L.Bsf, L.B, L.Bf);
  const SellV<T> NS = sv<T>(L.Ns, L.Nsf), GTS = sv<T>(L.GTs, L.GTsf), PS = sv<T>(L.Ps, L.Psf), PTS = sv<T>(L.PTs, L.PTsf),
                 PnS = sv<T>(L.Pns, L.Pnsf);
  const MatV<T> GT = view<T>(L.GT, L.GTf), PT = view<T>(L.PT, L.PTf), P = view<T>(L.P, L.Pf), Pn = view<T>(L.Pn, L.Pnf);
  const T *kd0 = arr<T>(L.kd[0], L.kdf[0]), *kd1 = arr<T>(L.kd[1], L.kdf[1]), *kd2 = arr<T>(L.kd[2], L.kdf[2]);
  const T *kl0 = arr<T>(L.kl[0], L.klf[0]), *kl1 = arr<T>(L.kl[1], L.klf[1]), *kl2 = arr<T>(L.kl[2], L.klf[2]);
  const T *nd0 = arr<T>(L.nd[0], L.ndf[0]), *nd1 = arr<T>(L.nd[1], L.ndf[1]);
  const T *nl0 = arr<T>(L.nl[0], L.nlf[0]), *nl1 = arr<T>(L.nl[1], L.nlf[1]);
  const T damp = (T)1.0;
  const unsigned ge = grid_rows(ne, k), gn = grid_rows(nn, k);
  // algorithmic bytes of one edge-kernel launch: K (columns + three values) and
  // its row pointers, B when phi is used, and each vector once
  KTimer *kt = (l == 0) ? w.kt : nullptr;
  auto edge_bytes = [&](int mode, int use_phi) {
    const double vb = (double)sizeof(C2<T>) * k, tb = (double)sizeof(T);
    const int kind = mode & EdgeMode::KIND;
    const bool use_k = !(mode & EdgeMode::NOK);
    double b = vb * ne * 2;                                                     // r in, out
    if (kind != EdgeMode::JACOBI0) {
      if (use_k) {
        b += (double)(L.K.nnz - L.K.nsdg) * (4 + L.K.nv * tb) + 8.0 * (ne + 1) + vb * ne;  // K, u
        if (L.K.dg[0]) b += 2 * tb * ne;                                        // diagonal K_eps, K_sig
        if (L.K.sdg) b += tb * ne;                                              // diagonal K_S
      }
      if (use_phi) b += (double)L.B.nnz * (4 + 2 * tb) + 8.0 * (ne + 1) + vb * nn;
    }
    if (kind != EdgeMode::RES) b += 6 * tb * ne;                                // smoother diagonals
    if (kind == EdgeMode::JACOBI && !use_k) b += vb * ne;                       // u for the update
    return b;
  };
  auto tb0 = [&]() { if (kt) kt->begin(s); };
  auto te0 = [&](int mode, int use_phi) { if (kt) kt->end(s, edge_bytes(mode, use_phi)); };
  // level-0 launches that gather K u go through the plane march when it applies
  auto edge = [&](const C2<T> *rr, const C2<T> *uu, const C2<T> *pp, C2<T> *oo, int mode, int use_phi, T dmp,
                  hipStream_t st) {
    if constexpr (std::is_same<T, float>::value) {
      if (l == 0 && w.edge_march &&
          edge_march(H, k, KS, BS, w.c1, w.c2, kd0, kd1, kd2, kl0, kl1, kl2, rr, uu, pp, oo, mode, use_phi, dmp, st))
        return;
    }
    edge_sell<T>(ne, w.sell_min_rows, k, KS, BS, K, B, w.c1, w.c2, kd0, kd1, kd2, kl0, kl1, kl2, rr, uu, pp, oo, mode,
                 use_phi, dmp, st);
  };
  // rn = G^T res and the nodal smoother's first sweep from zero, d = rn / d_n, in
  // one launch; where that sweep is the only one, sum += d with it (returned)
  // and rn stays in registers
  auto nodal_first = [&](C2<T> *d, C2<T> *sum, int nu) {
    if (nn == 0) return true;
    if (nn < w.sell_min_rows) {
      spmv_real_sell<T>(nn, w.sell_min_rows, k, GTS, GT, res, rn, 0, s);
      node_sell<T>(nn, w.sell_min_rows, k, NS, N, w.c1, w.c2, nd0, nd1, nl0, nl1, rn, nullptr, d, damp, s);
      return false;
    }
    Nod0<T> nz;
    nz.nd0 = nd0; nz.nd1 = nd1; nz.nl0 = nl0; nz.nl1 = nl1;
    nz.d = d; nz.damp = damp;
    nz.sum = nu == 1 ? sum : nullptr;
    spmv_real_sell<T, SPMV_NOD0>(nn, w.sell_min_rows, k, GTS, GT, res, nu == 1 ? nullptr : rn, 0, s, w.c1, w.c2, Jac0<T>(), nz);
    return nz.sum != nullptr;
  };
  // u and tmp trade places after every Jacobi sweep but the first; start from
  // the buffer that makes the last sweep write the level's own u (no copy)
  if (((nu_pre - 1) + nu_post) & 1) std::swap(u, tmp);
  if ((nu_pre - 1) & 1) std::swap(phi, d2);
  // pre-smoothing on the edges (phi = 0); the first sweep may have come out of
  // the pass that formed r (Jac0)
  if (w.u0_ready) {
    w.u0_ready = false;
  } else {
    tb0();
    edge(r, nullptr, nullptr, u, EdgeMode::JACOBI0, 0, damp, s);
    te0(EdgeMode::JACOBI0, 0);
  }
  for (int it = 1; it < nu_pre; ++it) {
    tb0();
    edge(r, u, nullptr, tmp, EdgeMode::JACOBI, 0, damp, s);
    te0(EdgeMode::JACOBI, 0);
    std::swap(u, tmp);
  }
  // pre-smoothing on the nodal auxiliary space
  tb0();
  edge(r, u, nullptr, res, EdgeMode::RES, 0, damp, s);
  te0(EdgeMode::RES, 0);
  nodal_first(phi, nullptr, nu_pre);
  for (int it = 1; it < nu_pre; ++it) {
    node_sell<T>(nn, w.sell_min_rows, k, NS, N, w.c1, w.c2, nd0, nd1, nl0, nl1, rn, phi, d2, damp, s);
    std::swap(phi, d2);
  }
  // coarse-grid correction.  res holds r - K u for this u already, so only
  // B phi is subtracted (no second K gather); the result goes to tmp, which
  // is free until the post-smoothing
  tb0();
  edge(res, u, phi, tmp, EdgeMode::RES | EdgeMode::NOK, 1, damp, s);
  te0(EdgeMode::RES | EdgeMode::NOK, 1);
  const int64_t nec = H.L[l + 1].ne, nnc = H.L[l + 1].nn;
  if (l + 2 < (int)H.L.size() && nec >= w.sell_min_rows) {  // with the next level's first sweep
    const MgLevel &C = H.L[l + 1];
    spmv_real_sell<T, SPMV_JAC0>(nec, w.sell_min_rows, k, PTS, PT, tmp, w.r[l + 1], 0, s, w.c1, w.c2,
                                 jac0_of<T>(C, w, l + 1, nu_pre, nu_post));
    w.u0_ready = nec > 0;
  } else {
    spmv_real_sell<T>(nec, w.sell_min_rows, k, PTS, PT, tmp, w.r[l + 1], 0, s);
  }
  GP_TRY(vcycle_level<T>(H, w, s, l + 1, nu_pre, nu_post));
  prolong_sell<T>(ne, nn, w.sell_min_rows, k, PS, P, w.u[l + 1], u, PnS, Pn, w.phi[l + 1], phi, s);
  (void)nnc;
  // post-smoothing: nodal, then edges
  tb0();
  edge(r, u, phi, res, EdgeMode::RES, 1, damp, s);
  te0(EdgeMode::RES, 1);
  const bool added = nodal_first(d1, phi, nu_post);
  for (int it = 1; it < nu_post; ++it) {
    node_sell<T>(nn, w.sell_min_rows, k, NS, N, w.c1, w.c2, nd0, nd1, nl0, nl1, rn, d1, d2, damp, s);
    std::swap(d1, d2);
  }
  if (!added) k_add<T><<<gn, 256, 0, s>>>(nn * k, phi, d1);
  for (int it = 0; it < nu_post; ++it) {
    // the first sweep starts from res = r - K u - B phi_old for this u: only
    // B d1 (the nodal correction just added to phi) is subtracted
    const int md = it == 0 ? (EdgeMode::JACOBI | EdgeMode::NOK) : EdgeMode::JACOBI;
    tb0();
    edge(it == 0 ? res : r, u, it == 0 ? d1 : phi, tmp, md, 1, damp, s);
    te0(md, 1);
    std::swap(u, tmp);
  }
  // results must land in the level's canonical buffers
  if (u != w.u[l]) GP_HIP(hipMemcpyAsync(w.u[l], u, sizeof(C2<T>) * ne * k, hipMemcpyDeviceToDevice, s));
  if (phi != w.phi[l]) GP_HIP(hipMemcpyAsync(w.phi[l], phi, sizeof(C2<T>) * nn * k, hipMemcpyDeviceToDevice, s));
  return GP_OK;
}

template <class T>
gp_status vcycle(const Hierarchy &H, VWork<T> &w, hipStream_t s, int nu_pre, int nu_post) {
  return vcycle_level<T>(H, w, s, 0, nu_pre, nu_post);
}

// Epilogue of the product that forms level l's right-hand side: the level's
// first sweep from zero with it (into the buffer aux_cycle starts from), except
// on the coarsest level.
template <class T>
AuxEp<T> aux_first(const AuxAMG &X, const VWork<T> &w, int l) {
  AuxEp<T> ep;
  ep.y = w.ar[l];
  if (l + 1 < (int)X.L.size()) {
    const AuxLevel &L = X.L[l];
    ep.z = w.at[l];
    ep.d0 = arr<T>(L.nd[0], L.ndf[0]); ep.d1 = arr<T>(L.nd[1], L.ndf[1]);
    ep.l0 = arr<T>(L.nl[0], L.nlf[0]); ep.l1 = arr<T>(L.nl[1], L.nlf[1]);
  }
  return ep;
}

// Auxiliary AMG V-cycle on level l: input w.ar[l] and its first sweep
// (aux_first), output w.ax[l].
template <class T>
static gp_status aux_cycle(const Hierarchy &H, VWork<T> &w, hipStream_t s, int l) {
  const AuxAMG &X = H.aux;
  const AuxLevel &L = X.L[l];
  const int k = w.k;
  const int64_t n = L.n;
  C2<T> *r = w.ar[l], *x = w.ax[l], *t = w.at[l];
  if (l + 1 == (int)X.L.size()) {
    if (X.eig) return aux_eig_apply<T>(X, k, w.om64, r, x, w.eig_y, s);
    k_blkdiag_apply<T><<<dim3((unsigned)((n + 3) / 4), (unsigned)k), 256, 0, s>>>(n, k, X.perm, X.rowblk, X.boff,
                                                                                 X.ioff, w.fidx, w.tab + 3 * w.cap, r, x);
    return GP_OK;
  }
  const MatV<T> N = view<T>(L.N, L.Nf), P = view<T>(L.P, L.Pf), PT = view<T>(L.PT, L.PTf);
  const SellV<T> NS = sv<T>(L.Ns, L.Nsf), PS = sv<T>(L.Ps, L.Psf), PTS = sv<T>(L.PTs, L.PTsf);
  const T *d0 = arr<T>(L.nd[0], L.ndf[0]), *d1 = arr<T>(L.nd[1], L.ndf[1]);
  const T *l0 = arr<T>(L.nl[0], L.nlf[0]), *l1 = arr<T>(L.nl[1], L.nlf[1]);
  const int nu = w.nu_aux;
  // x and t trade places after every sweep but the first (2 nu - 1 swaps):
  // start from t so that the last sweep writes the level's own x.  The first
  // sweep from zero came with r (aux_first, from the product that formed it)
  std::swap(x, t);
  AuxEp<T> jac;
  jac.r = r; jac.d0 = d0; jac.d1 = d1; jac.l0 = l0; jac.l1 = l1;
  auto sweep = [&]() {
    jac.y = t;
    aux_prod<T, AX_JAC>(n, w, NS, N, x, jac, s);
    std::swap(x, t);
  };
  for (int it = 1; it < nu; ++it) sweep();
  AuxEp<T> res;
  res.r = r; res.y = t;
  aux_prod<T, AX_RES>(n, w, NS, N, x, res, s);
  aux_prod<T, AX_REAL>(X.L[l + 1].n, w, PTS, PT, t, aux_first<T>(X, w, l + 1), s);
  GP_TRY(aux_cycle<T>(H, w, s, l + 1));
  AuxEp<T> add;
  add.y = x; add.accumulate = 1;
  aux_prod<T, AX_REAL>(n, w, PS, P, w.ax[l + 1], add, s);
  for (int it = 0; it < nu; ++it) sweep();
  if (x != w.ax[l]) GP_HIP(hipMemcpyAsync(w.ax[l], x, sizeof(C2<T>) * n * k, hipMemcpyDeviceToDevice, s));
  return GP_OK;
}

template <class T>
gp_status precond(const Hierarchy &H, VWork<T> &w, hipStream_t s, int nu_pre, int nu_post) {
  const AuxAMG &X = H.aux;
  const MgLevel &L0 = H.L[0];
  const int k = w.k;
  const int64_t n = L0.ne, na = X.naux;
  const MatV<T> GxT = view<T>(X.GxT, X.GxTf), Bx = view<T>(X.Bx, X.Bxf);
  const SellV<T> GxTS = sv<T>(X.GxTs, X.GxTsf), BxS = sv<T>(X.Bxs, X.Bxsf);
  const MatV<T> K = view<T>(L0.K, L0.Kf), B = view<T>(L0.B, L0.Bf);
  const unsigned gn = grid_rows(n, k), ga = grid_rows(na, k);
  // auxiliary correction: a = AMG(Gx^T r), r <- r - Bx a
  if (w.aux_post) k_copy<T><<<blocks_for(n * k), 256, 0, s>>>(n * k, w.r[0], w.r0);
  aux_prod<T, AX_REAL>(na, w, GxTS, GxT, w.r[0], aux_first<T>(X, w, 0), s);
  if (w.aux_post) {
    GP_TRY(aux_cycle<T>(H, w, s, 0));
    k_copy<T><<<blocks_for(na * k), 256, 0, s>>>(na * k, w.ax[0], w.a);
  } else {
    // one-sided form: the cycle's level-0 result lands in w.a directly
    C2<T> *ax0 = w.ax[0];
    w.ax[0] = w.a;
    const gp_status ast = aux_cycle<T>(H, w, s, 0);
    w.ax[0] = ax0;
    GP_TRY(ast);
  }
  // the edge V-cycle's first level-0 sweep (u = r / d_l1 from zero) comes out
  // of the same pass, into the buffer that sweep would write
  Jac0<T> jz;
  if (H.L.size() > 1) jz = jac0_of<T>(L0, w, 0, nu_pre, nu_post);
  w.u0_ready = spmv2_sell<T>(n, w.sell_min_rows, k, BxS, Bx, w.c1, w.c2, w.a, w.r[0], s, jz);
  // edge V-cycle on the remaining residual
  GP_TRY(vcycle<T>(H, w, s, nu_pre, nu_post));
  // The second auxiliary correction (on r0 - K u - B phi - Bx a) makes the
  // preconditioner symmetric; FGMRES does not need that, and without it each
  // application skips a level-0 residual, the Bx / Gx^T products and one
  // auxiliary cycle.  Measured at 200x200x24, 80 columns: 18.3 solves/s
  // without it (iterations p50 44, max 126) against 17.2 with it (37, 103),
  // per-column latency p50 0.69 s / p99 1.99 s against 0.75 s / 2.10 s.
  if (!w.aux_post) return GP_OK;
  const T *kd0 = arr<T>(L0.kd[0], L0.kdf[0]);
  (void)kd0;
  const SellV<T> KS = sview<T>(L0.Ks, L0.Ksf, L0.K, L0.Kf), BS = sview<T>(L0.Bs, L0.Bsf, L0.B, L0.Bf);
  bool marched = false;
  if constexpr (std::is_same<T, float>::value)
    marched = w.edge_march && edge_march(H, k, KS, BS, w.c1, w.c2, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                                         w.r0, w.u[0], w.phi[0], w.res[0], EdgeMode::RES, 1, 1.0f, s);
  if (!marched)
    edge_sell<T>(n, w.sell_min_rows, k, KS, BS, K, B, w.c1, w.c2, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                 w.r0, w.u[0], w.phi[0], w.res[0], EdgeMode::RES, 1, (T)1, s);
  spmv2_sell<T>(n, w.sell_min_rows, k, BxS, Bx, w.c1, w.c2, w.a, w.res[0], s);
  aux_prod<T, AX_REAL>(na, w, GxTS, GxT, w.res[0], aux_first<T>(X, w, 0), s);
  GP_TRY(aux_cycle<T>(H, w, s, 0));
  k_add<T><<<blocks_for(na * k), 256, 0, s>>>(na * k, w.a, w.ax[0]);
  return GP_OK;
}

template gp_status precond<float>(const Hierarchy &, VWork<float> &, hipStream_t, int, int);
template gp_status precond<double>(const Hierarchy &, VWork<double> &, hipStream_t, int, int);

template gp_status vwork_create<float>(gp_layout *, const Hierarchy &, int, VWork<float> *);
template gp_status vwork_create<double>(gp_layout *, const Hierarchy &, int, VWork<double> *);
template gp_status vwork_set_columns<float>(VWork<float> &, const double *, const int32_t *, const CoarseCache &, hipStream_t);
template gp_status vwork_set_columns<double>(VWork<double> &, const double *, const int32_t *, const CoarseCache &, hipStream_t);
template void vwork_free<float>(VWork<float> *);
template void vwork_free<double>(VWork<double> *);
template gp_status vcycle<float>(const Hierarchy &, VWork<float> &, hipStream_t, int, int);
template gp_status vcycle<double>(const Hierarchy &, VWork<double> &, hipStream_t, int, int);

int set_lanes_cap(int cap) {
  const int prev = t_lanes_cap;
  if (cap >= 1) t_lanes_cap = cap;
  return prev;
}

}  // namespace gp

// dense.hip -- dense FP64 inverses (Gauss-Jordan, partial pivoting) of the
// coarsest multigrid levels: complex ones, one matrix per frequency, and the
// real AMG's.
//
// A matrix is inverted in place of its own n x n array (no augmentation): an
// elimination step exchanges an unknown with a right-hand side, so step c
// leaves column c of the inverse where column c of the matrix was.  Rows are
// not swapped; rc[c] records the pivot row of column c and the last kernel
// puts rows and columns in order.  k_gj_panel takes up to eight steps per
// launch (see there); matrices of which not even two columns fit a workgroup's
// LDS (more than ~1900 complex or ~3700 real rows) take a launch per step.
//
// Blocks of the auxiliary coarsest level without its eigenvector form are many
// and small: one workgroup each, all in one launch (k_gj_block).
#include <cmath>

#include "dense.hpp"

namespace gp {

namespace {

typedef C2<double> Z2;

__device__ __forceinline__ double gj_abs2(double v) { return v * v; }
__device__ __forceinline__ double gj_abs2(const Z2 &v) { return v.x * v.x + v.y * v.y; }
__device__ __forceinline__ double gj_inv(double v) { return 1.0 / v; }
__device__ __forceinline__ Z2 gj_inv(const Z2 &v) {
  const double d = v.x * v.x + v.y * v.y;
  return {v.x / d, -v.y / d};
}
__device__ __forceinline__ double gj_mul(double a, double b) { return a * b; }
__device__ __forceinline__ Z2 gj_mul(const Z2 &a, const Z2 &b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
__device__ __forceinline__ void gj_sub(double &x, double a, double b) { x -= a * b; }
__device__ __forceinline__ void gj_sub(Z2 &x, const Z2 &a, const Z2 &b) {
  x.x -= a.x * b.x - a.y * b.y;
  x.y -= a.x * b.y + a.y * b.x;
}
__device__ __forceinline__ double gj_neg(double a) { return -a; }
__device__ __forceinline__ Z2 gj_neg(const Z2 &a) { return {-a.x, -a.y}; }
template <class Z> __device__ __forceinline__ Z gj_zero();
template <> __device__ __forceinline__ double gj_zero<double>() { return 0.; }
template <> __device__ __forceinline__ Z2 gj_zero<Z2>() { return {0., 0.}; }

// (value, row) of the larger value over the workgroup, ties to the smaller
// row; every thread gets it
__device__ __forceinline__ void gj_argmax(double &v, int &r, double *sv, int *si) {
  for (int o = 32; o > 0; o >>= 1) {
    const double ov = __shfl_xor(v, o);
    const int orow = __shfl_xor(r, o);
    if (ov > v || (ov == v && orow < r)) { v = ov; r = orow; }
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { sv[wave] = v; si[wave] = r; }
  __syncthreads();
  v = sv[0];
  r = si[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
    if (sv[w] > v || (sv[w] == v && si[w] < r)) { v = sv[w]; r = si[w]; }
}

// Whether matrix b was found singular, the same answer for the whole workgroup.
// Workgroups of one launch reach that verdict at different times, so one thread
// reads the flag: were each wavefront to read it, some would leave and the rest
// pick a pivot from LDS slots that nobody wrote.
__device__ __forceinline__ bool gj_gone(const int *bad, int b, int *flag) {
  if (threadIdx.x == 0) *flag = __hip_atomic_load(bad + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  return *flag != 0;
}

constexpr int kGJPanel = 8;   // most elimination steps per launch
constexpr int kGJTile = 8;    // columns per workgroup

// The m = min(M, n - c0) elimination steps of columns c0 .. c0 + m - 1, src ->
// dst.  Every workgroup runs the steps on the n x m panel in LDS (the same
// arithmetic in each: a few hundred rows, so repeating it costs less than a
// launch per step and one more for its pivot), then updates its kGJTile
// columns with the m pivot rows at once.  Grid (column tiles, matrices).
// One workgroup walking all n steps over the whole matrix (the layout before)
// ran at the speed of one CU: 51 ms for the 471-row coarsest level of
// real AMG at 128x128x16, 1.7 ms now (59 launches).
template <class Z, int M>
__global__ void __launch_bounds__(256) k_gj_panel(int n, int c0, const Z *__restrict__ src_, Z *__restrict__ dst_,
                                                  int32_t *__restrict__ rc_, int *bad) {
  extern __shared__ double2 gj_lds[];
  __shared__ double sv[4];
  __shared__ int si[4], gone;
  __shared__ int prow[M];
  __shared__ Z piv[M];
  __shared__ Z X[M][kGJTile];
  const int m = min(M, n - c0);
  Z *P = reinterpret_cast<Z *>(gj_lds);                             // column q at q n: a wavefront's rows in a line
  unsigned char *used = reinterpret_cast<unsigned char *>(P + (int64_t)n * M);  // n
  const int b = blockIdx.y, tid = threadIdx.x;
  if (gj_gone(bad, b, &gone)) return;
  const Z *src = src_ + (int64_t)b * n * n;
  Z *dst = dst_ + (int64_t)b * n * n;
  int32_t *rc = rc_ + (int64_t)b * n;
  for (int r = tid; r < n; r += 256) used[r] = 0;
  __syncthreads();
  for (int c = tid; c < c0; c += 256) used[rc[c]] = 1;
  // past the last column: zeros, which the steps leave alone
#pragma unroll 8
  for (int t = tid; t < n * M; t += 256) P[(t % M) * n + t / M] = t % M < m ? src[(int64_t)(t / M) * n + c0 + t % M] : gj_zero<Z>();
  __syncthreads();
  for (int q = 0; q < m; ++q) {
    double best = -1.0;
    int p = n;
    for (int r = tid; r < n; r += 256) {
      if (used[r]) continue;
      const double v = gj_abs2(P[q * n + r]);
      if (v > best) { best = v; p = r; }
    }
    gj_argmax(best, p, sv, si);
    if (!(best > 0.0)) {  // the same for every thread: the workgroup leaves together
      if (tid == 0) bad[b] = 1;
      return;
    }
    if (tid < M) piv[tid] = P[tid * n + p];
    if (tid == 0) { used[p] = 1; prow[q] = p; }
    __syncthreads();
    const Z d = gj_inv(piv[q]);
    Z pv[M];
#pragma unroll
    for (int t = 0; t < M; ++t) pv[t] = piv[t];
    for (int r = tid; r < n; r += 256) {
      Z x[M];
#pragma unroll
      for (int t = 0; t < M; ++t) x[t] = P[t * n + r];
      const Z g = gj_mul(P[q * n + r], d);
#pragma unroll
      for (int t = 0; t < M; ++t) {
        if (r == p) x[t] = gj_neg(gj_mul(pv[t], d));
        else gj_sub(x[t], g, pv[t]);
        P[t * n + r] = x[t];
      }
      P[q * n + r] = r == p ? d : g;
    }
    __syncthreads();
  }
  const int j0 = blockIdx.x * kGJTile;
  if (blockIdx.x == 0 && tid < m) rc[c0 + tid] = prow[tid];
  if (tid < M * kGJTile) {
    const int q = tid / kGJTile, j = j0 + tid % kGJTile;
    X[q][tid % kGJTile] = j < n && q < m ? src[(int64_t)prow[q] * n + j] : gj_zero<Z>();
    if (q >= m && tid % kGJTile == 0) prow[q] = -1;
  }
  __syncthreads();
  const int jj = tid % kGJTile, j = j0 + jj;
  if (j >= n) return;
#pragma unroll 4
  for (int r = tid / kGJTile; r < n; r += 256 / kGJTile) {
    Z x;
    if (j >= c0 && j < c0 + m) {
      x = P[(j - c0) * n + r];
    } else {
      bool pr = false;
#pragma unroll
      for (int q = 0; q < M; ++q) pr = pr || prow[q] == r;
      x = pr ? gj_zero<Z>() : src[(int64_t)r * n + j];
#pragma unroll
      for (int q = 0; q < M; ++q) gj_sub(x, P[q * n + r], X[q][jj]);
    }
    dst[(int64_t)r * n + j] = x;
  }
}

// One elimination step of column c, src -> dst (matrices too tall for a panel
// in LDS): every workgroup finds the pivot of the column itself, then updates
// its rows.  Grid (row tiles, matrices).
template <class Z>
__global__ void __launch_bounds__(256) k_gj_step(int n, int c, const Z *__restrict__ src_, Z *__restrict__ dst_,
                                                 int32_t *__restrict__ rc_, int32_t *__restrict__ used_,
                                                 int *bad) {
  __shared__ double sv[4];
  __shared__ int si[4], gone;
  const int b = blockIdx.y, tid = threadIdx.x;
  if (gj_gone(bad, b, &gone)) return;
  const Z *src = src_ + (int64_t)b * n * n;
  Z *dst = dst_ + (int64_t)b * n * n;
  // used[r]: one more than the step that took row r (0: none yet); this step's
  // mark is written by one workgroup and ignored by the others
  int32_t *used = used_ + (int64_t)b * n;
  double best = -1.0;
  int p = n;
  for (int r = tid; r < n; r += 256) {
    const int u = used[r];
    if (u != 0 && u != c + 1) continue;
    const double v = gj_abs2(src[(int64_t)r * n + c]);
    if (v > best) { best = v; p = r; }
  }
  gj_argmax(best, p, sv, si);
  if (!(best > 0.0)) {
    if (tid == 0) bad[b] = 1;
    return;
  }
  if (blockIdx.x == 0 && tid == 0) { rc_[(int64_t)b * n + c] = p; used[p] = c + 1; }
  const Z d = gj_inv(src[(int64_t)p * n + c]);
  const int r0 = blockIdx.x * 16;
  for (int r = r0; r < min(n, r0 + 16); ++r) {
    const Z f = gj_mul(src[(int64_t)r * n + c], d);
    for (int j = tid; j < n; j += 256) {
      Z x;
      if (r == p) x = j == c ? d : gj_neg(gj_mul(src[(int64_t)p * n + j], d));
      else if (j == c) x = f;
      else { x = src[(int64_t)r * n + j]; gj_sub(x, f, src[(int64_t)p * n + j]); }
      dst[(int64_t)r * n + j] = x;
    }
  }
}

// the inverse from the exchanged tableau: row rc[i] belongs to unknown i,
// column c to right-hand side rc[c]
template <class Z>
__global__ void k_gj_order(int n, int nb, const Z *__restrict__ t_, const int32_t *__restrict__ rc_, Z *__restrict__ a_) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (int64_t)nb * n * n) return;
  const int64_t b = t / ((int64_t)n * n), rem = t - b * n * n;
  const int64_t i = rem / n, c = rem - i * n;
  const int32_t *rc = rc_ + b * n;
  a_[(b * n + i) * n + rc[c]] = t_[(b * n + rc[i]) * n + c];
}

// Gauss-Jordan with partial pivoting on one augmented matrix [A | I] per
// workgroup (at most kGJWorkgroupMax rows), in device memory: the blocks in
// `list`, each in L2 while its steps, ordered by the workgroup's barriers, run.
// bad[0] is set if a pivot column is exactly zero.
__global__ void __launch_bounds__(1024) k_gj_block(const int32_t *__restrict__ list, const int32_t *__restrict__ boff,
                                                   const int64_t *__restrict__ aoff, C2<double> *__restrict__ aug,
                                                   int *__restrict__ bad) {
  __shared__ double sv[1024];
  __shared__ int si[1024];
  __shared__ C2<double> fcol[kGJWorkgroupMax];
  const int blk = list[blockIdx.x];
  const int b = boff[blk + 1] - boff[blk];
  C2<double> *A = aug + aoff[blk];
  const int w = 2 * b;
  const int tid = threadIdx.x, nt = blockDim.x;
  for (int c = 0; c < b; ++c) {
    double best = -1.0;
    int bi = c;
    for (int r = c + tid; r < b; r += nt) {
      const C2<double> v = A[r * w + c];
      const double m = v.x * v.x + v.y * v.y;
      if (m > best) { best = m; bi = r; }
    }
    sv[tid] = best;
    si[tid] = bi;
    __syncthreads();
    for (int h = nt / 2; h > 0; h >>= 1) {
      if (tid < h) {
        const double o = sv[tid + h];
        const int oi = si[tid + h];
        if (o > sv[tid] || (o == sv[tid] && oi < si[tid])) { sv[tid] = o; si[tid] = oi; }
      }
      __syncthreads();
    }
    const int piv = si[0];
    if (!(sv[0] > 0.0)) {              // the same value for every thread: all leave together
      if (tid == 0) bad[0] = 1;
      return;
    }
    if (piv != c)
      for (int j = c + tid; j < w; j += nt) {
        const C2<double> t = A[c * w + j];
        A[c * w + j] = A[piv * w + j];
        A[piv * w + j] = t;
      }
    __syncthreads();
    const C2<double> p = A[c * w + c];
    const double d = p.x * p.x + p.y * p.y;
    const C2<double> inv = {p.x / d, -p.y / d};
    __syncthreads();
    for (int j = c + tid; j < w; j += nt) {
      const C2<double> v = A[c * w + j];
      A[c * w + j] = {v.x * inv.x - v.y * inv.y, v.x * inv.y + v.y * inv.x};
    }
    __syncthreads();
    for (int r = tid; r < b; r += nt) fcol[r] = A[r * w + c];
    __syncthreads();
    const int wc = w - c;
    for (int t = tid; t < b * wc; t += nt) {
      const int r = t / wc, j = c + (t - r * wc);
      if (r == c) continue;
      const C2<double> f = fcol[r], v = A[c * w + j];
      C2<double> x = A[r * w + j];
      x.x -= f.x * v.x - f.y * v.y;
      x.y -= f.x * v.y + f.y * v.x;
      A[r * w + j] = x;
    }
    __syncthreads();
  }
}

}  // namespace

gp_status gj_workgroup(const int32_t *list, const int32_t *boff, const int64_t *aoff, int count, C2<double> *aug,
                       int *bad, hipStream_t s) {
  if (count <= 0) return GP_OK;
  k_gj_block<<<count, 1024, 0, s>>>(list, boff, aoff, aug, bad);
  GP_HIP(hipGetLastError());
  return GP_OK;
}

namespace {

template <class Z>
gp_status inverse(Z *a, int n, int nb, hipStream_t s) {
  if (n <= 0 || nb <= 0) return GP_OK;
  TmpArena T;
  struct Free { Arena &a; hipStream_t s; ~Free() { (void)hipStreamSynchronize(s); a.free_all(); } } fr{T, s};
  Z *t0 = nullptr, *t1 = nullptr;
  int32_t *rc = nullptr, *used = nullptr;
  int *bad = nullptr;
  GP_TRY(T.alloc(&t0, (int64_t)nb * n * n)); GP_TRY(T.alloc(&t1, (int64_t)nb * n * n));
  GP_TRY(T.alloc(&rc, (int64_t)nb * n)); GP_TRY(T.alloc(&bad, (int64_t)nb));
  GP_HIP(hipMemsetAsync(bad, 0, sizeof(int) * nb, s));
  // the widest panel that fits 64 KB of LDS beside the workgroup's small arrays
  int M = kGJPanel;
  while (M > 1 && (int64_t)n * M * (int64_t)sizeof(Z) + n + 1600 > 65536) M >>= 1;
  const Z *src = a;
  Z *dst = t0;
  if (M > 1) {
    const size_t shm = (size_t)n * M * sizeof(Z) + n;
    const dim3 grid((unsigned)((n + kGJTile - 1) / kGJTile), (unsigned)nb);
    for (int c = 0; c < n; c += M) {
      if (M == 8) k_gj_panel<Z, 8><<<grid, 256, shm, s>>>(n, c, src, dst, rc, bad);
      else if (M == 4) k_gj_panel<Z, 4><<<grid, 256, shm, s>>>(n, c, src, dst, rc, bad);
      else k_gj_panel<Z, 2><<<grid, 256, shm, s>>>(n, c, src, dst, rc, bad);
      src = dst;
      dst = dst == t0 ? t1 : t0;
    }
  } else {
    GP_TRY(T.alloc(&used, (int64_t)nb * n));
    GP_HIP(hipMemsetAsync(used, 0, sizeof(int32_t) * nb * n, s));
    const dim3 grid((unsigned)((n + 15) / 16), (unsigned)nb);
    for (int c = 0; c < n; ++c) {
      k_gj_step<Z><<<grid, 256, 0, s>>>(n, c, src, dst, rc, used, bad);
      src = dst;
      dst = dst == t0 ? t1 : t0;
    }
  }
  GP_HIP(hipGetLastError());
  std::vector<int> hb(nb);
  GP_HIP(hipMemcpyAsync(hb.data(), bad, sizeof(int) * nb, hipMemcpyDeviceToHost, s));
  GP_HIP(hipStreamSynchronize(s));
  for (int b = 0; b < nb; ++b)
    if (hb[b]) return fail(GP_ERR_ARG, "singular coarsest-level matrix");
  k_gj_order<Z><<<blocks_for((int64_t)nb * n * n), 256, 0, s>>>(n, nb, src, rc, a);
  GP_HIP(hipGetLastError());
  return GP_OK;
}

}  // namespace

gp_status dense_inverse_batched(C2<double> *a, int n, int nb, hipStream_t s) { return inverse<Z2>(a, n, nb, s); }
gp_status dense_inverse_real(double *a, int n, hipStream_t s) { return inverse<double>(a, n, 1, s); }

}  // namespace gp

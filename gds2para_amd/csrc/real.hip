// real.hip -- real sparse solve replacing hypreSolve (src/hypreSolve.cpp:9-283,
// interface src/hypreSolver.h:14): A x = b for a real matrix given as
// row-sorted COO triplets, by flexible GMRES(30) in FP64 preconditioned with
// one V-cycle of smoothed-aggregation AMG built from the matrix alone.
//
// The reference runs HYPRE FlexGMRES (KDim 10, max 100 iterations, relative
// tolerance 1e-4) with BoomerAMG.  Here the tolerance is the caller's (1e-4
// when 0 is passed, the reference's value) and the AMG is:
//   * aggregation: two passes of strength-weighted pairwise matching (each
//     node pairs with its strongest unmatched strong neighbour when the
//     choice is mutual; j is a strong neighbour of i when
//     |a_ij| / sqrt|a_ii a_jj| is at least kTheta of the row's largest such
//     score), so aggregates hold up to four nodes;
//   * prolongation: the aggregates' indicator smoothed once with
//     4/(3 lambda) D^-1 A (lambda from power iteration), truncated (entries
//     below kTrunc of the row's largest dropped, the row's own aggregate
//     kept, the row sum restored), Galerkin R A P;
//   * smoothing, two matrix products each side: l1-Jacobi sweeps (the
//     default) or two steps of the Chebyshev recurrence on D^-1 A over
//     [0.3 b, b], b = 1.1 lambda (gp_solve_real_ex; the reference picks
//     BoomerAMG's relaxation with HYPRE_BoomerAMGSetRelaxType,
//     src/hypreSolve.cpp:230); dense FP64 inverse on the coarsest level
//     (<= 512 unknowns).
// A solve takes 1, 2, 4 or 8 right-hand sides side by side (vectors
// interleaved, row i column j at i*K + j): every matrix entry and every launch
// serves all of them, while each column keeps its own recurrence.
#include <algorithm>
#include <cmath>
#include <complex>
#include <vector>

#include "dense.hpp"
#include "real.hpp"
#include "sparse.hpp"

namespace gp {

namespace {

constexpr double kTheta = 0.25;
constexpr double kTrunc = 0.2;
constexpr int64_t kCoarsest = 512;
// Chebyshev smoothing: steps per side (the matrix products of two Jacobi
// sweeps) and its interval [kChebLower b, b] on the spectrum of D^-1 A, with
// b = kChebUpper times the power-iteration estimate of its largest eigenvalue
// (the estimate approaches it from below)
constexpr int kChebSteps = 2;
constexpr double kChebUpper = 1.1;
constexpr double kChebLower = 0.3;

// The setup kernels below give each row one wavefront (kWave lanes striding
// over its entries): Ad's conductor-aggregate rows couple to every dielectric
// node around a conductor, and one thread per row left each launch waiting
// on those few rows.  The wavefronts stride over the rows, so any n fits the
// grid of wave_blocks(n).
constexpr int kWave = 64;

unsigned wave_blocks(int64_t n) {
  return (unsigned)std::min<int64_t>(std::max<int64_t>((n * kWave + 255) / 256, 1), 1 << 20);
}

__device__ __forceinline__ int64_t wave_first() { return ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave; }
__device__ __forceinline__ int64_t wave_count() { return ((int64_t)gridDim.x * blockDim.x) / kWave; }

__device__ __forceinline__ double wave_sum(double x) {
  for (int o = kWave / 2; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}

__device__ __forceinline__ double wave_max(double x) {
  for (int o = kWave / 2; o > 0; o >>= 1) x = fmax(x, __shfl_xor(x, o));
  return x;
}

__global__ void k_r_diag(int64_t n, const int64_t *__restrict__ rp, const int32_t *__restrict__ ci,
                         const double *__restrict__ v, double *__restrict__ d, double *__restrict__ dl1) {
  const int lane = threadIdx.x & (kWave - 1);
  for (int64_t i = wave_first(); i < n; i += wave_count()) {  // i is the same on every lane
    double a = 0., off = 0.;
    for (int64_t p = rp[i] + lane; p < rp[i + 1]; p += kWave) {
      if (ci[p] == (int32_t)i) a += v[p];
      else off += fabs(v[p]);
    }
    a = wave_sum(a);
    off = wave_sum(off);
    if (lane == 0) {
      d[i] = a;
      const double m = fabs(a);
      dl1[i] = m > 0 ? a * (1.0 + off / m) : (off > 0 ? off : 1.0);
    }
  }
}

// symmetric perturbation in [1, 1 + 2^-10) of the strength of edge {i, j}:
// with equal strengths (a uniform grid) the heaviest edge at a node is then
// also the heaviest at its partner, so picks are mutual (locally dominant
// edge matching) instead of chaining along the index order
__device__ __forceinline__ double edge_jitter(int64_t i, int64_t j) {
  const uint64_t a = (uint64_t)(i < j ? i : j), b = (uint64_t)(i < j ? j : i);
  uint64_t h = a * 0x9E3779B97F4A7C15ULL ^ (b + 0x632BE59BD9B4E019ULL + (a << 6) + (a >> 2));
  h ^= h >> 31; h *= 0xBF58476D1CE4E5B9ULL; h ^= h >> 27;
  return 1.0 + (double)(h >> 11) * (1.0 / 9007199254740992.0) * (1.0 / 1024.0);
}

// each unmatched node picks its strongest unmatched strong neighbour (the
// largest jittered score, the smallest index among equal ones: max and the
// comparisons are exact, so the lanes' partial picks combine to the pick of
// one pass over the row)
__global__ void k_pick(int64_t n, const int64_t *__restrict__ rp, const int32_t *__restrict__ ci,
                       const double *__restrict__ v, const double *__restrict__ d, const int32_t *__restrict__ matched,
                       int32_t *__restrict__ pick) {
  const int lane = threadIdx.x & (kWave - 1);
  for (int64_t i = wave_first(); i < n; i += wave_count()) {  // i is the same on every lane
    int32_t best = -1;
    double bs = 0.;
    if (!matched[i]) {
      const int64_t b = rp[i], e = rp[i + 1];
      double rmax = 0.;
      for (int64_t p = b + lane; p < e; p += kWave) {
        const int32_t j = ci[p];
        if (j == (int32_t)i) continue;
        const double den = sqrt(fabs(d[i] * d[j]));
        rmax = fmax(rmax, den > 0 ? fabs(v[p]) / den : 0.);
      }
      const double thr = kTheta * wave_max(rmax);
      for (int64_t p = b + lane; p < e; p += kWave) {
        const int32_t j = ci[p];
        if (j == (int32_t)i || matched[j]) continue;
        const double den = sqrt(fabs(d[i] * d[j]));
        const double sc0 = den > 0 ? fabs(v[p]) / den : 0.;
        if (!(sc0 > 0.) || sc0 < thr) continue;
        const double sc = sc0 * edge_jitter(i, j);
        if (sc > bs || (sc == bs && j < best)) { bs = sc; best = j; }
      }
      for (int o = kWave / 2; o > 0; o >>= 1) {
        const double s2 = __shfl_xor(bs, o);
        const int32_t j2 = __shfl_xor(best, o);
        if (s2 > bs || (s2 == bs && j2 < best)) { bs = s2; best = j2; }
      }
    }
    if (lane == 0) pick[i] = best;
  }
}

// mutual picks become pairs
__global__ void k_pair(int64_t n, const int32_t *__restrict__ pick, int32_t *__restrict__ partner,
                       int32_t *__restrict__ matched_next) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int32_t j = pick[i];
  if (j >= 0 && pick[j] == (int32_t)i) { partner[i] = j; matched_next[i] = 1; }
}

__global__ void k_copy_i32(int64_t n, const int32_t *__restrict__ a, int32_t *__restrict__ b) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i];
}

__global__ void k_roots(int64_t n, const int32_t *__restrict__ partner, int64_t *__restrict__ root) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  root[i] = (partner[i] < 0 || (int32_t)i < partner[i]) ? 1 : 0;
}

// tentative prolongation: row i has one entry 1 in its aggregate's column
__global__ void k_ptent_pairs(int64_t n, const int32_t *__restrict__ partner, const int64_t *__restrict__ rootscan,
                              int64_t *__restrict__ rp, int32_t *__restrict__ ci, double *__restrict__ v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i > n) return;
  rp[i] = i;
  if (i == n) return;
  const int32_t q = partner[i];
  const int64_t r = (q < 0 || (int32_t)i < q) ? i : q;
  ci[i] = (int32_t)rootscan[r];
  v[i] = 1.0;
}

__global__ void k_r_dinv_spmv(int64_t n, const int64_t *__restrict__ rp, const int32_t *__restrict__ ci,
                              const double *__restrict__ v, const double *__restrict__ d, const double *__restrict__ x,
                              double *__restrict__ y) {
  const int lane = threadIdx.x & (kWave - 1);
  for (int64_t i = wave_first(); i < n; i += wave_count()) {  // i is the same on every lane
    double s = 0.;
    for (int64_t p = rp[i] + lane; p < rp[i + 1]; p += kWave) s += v[p] * x[ci[p]];
    s = wave_sum(s);
    if (lane == 0) y[i] = d[i] != 0. ? s / d[i] : 0.;
  }
}

// rows of A scaled by f / d_i (the smoothing matrix of the prolongation)
__global__ void k_r_scale_rows(int64_t n, int64_t nnz, const int64_t *__restrict__ rp, const double *__restrict__ v,
                               const double *__restrict__ d, double f, double *__restrict__ out) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nnz) return;
  const double di = d[csr_row_of(rp, n, p)];
  out[p] = (di != 0. ? f / di : 0.) * v[p];
}

// ---------------------------------------------------------------- products of K columns

// One row product s = sum a x of K columns and what is done with it:
//   R_MUL:  y = alpha s (+ y); with z also the first sweep of y's level from
//           zero, z = q, dd = q (if given) with q = zc y / zd
//   R_RES:  y = r - s
//   R_JAC:  y = x + (r - s) / d                      (l1-Jacobi, d = l1 diagonal)
//   R_CHEB: q = c2 (r - s) / d + c1 dd;  dd = q;  y = x + q
// (Chebyshev smoothing, the three-term recurrence written with a direction
// vector dd, Saad, Iterative Methods for Sparse Linear Systems, 2nd ed., Alg.
// 12.1, preconditioned with D^-1; c1 = 0 starts the recurrence from a nonzero
// x, dd is then not read).  y may be r.
enum RMode { R_MUL = 0, R_RES = 1, R_JAC = 2, R_CHEB = 3 };

struct REp {
  double *y = nullptr;
  const double *r = nullptr;
  double alpha = 1.;
  int acc = 0;
  const double *d = nullptr;
  double c1 = 0., c2 = 0.;
  double *dd = nullptr;
  double *z = nullptr;
  const double *zd = nullptr;
  double zc = 0.;
};

template <int K, int MODE>
__device__ __forceinline__ void r_row(const REp &ep, const double *x, int64_t i, int c, double s) {
  const int64_t q = i * K + c;
  if (MODE == R_MUL) {
    double v = ep.alpha * s;
    if (ep.acc) v = ep.y[q] + v;
    ep.y[q] = v;
    if (ep.z) {
      const double d = ep.zd[i], f = d != 0. ? ep.zc * v / d : 0.;
      ep.z[q] = f;
      if (ep.dd) ep.dd[q] = f;
    }
  } else if (MODE == R_RES) {
    ep.y[q] = ep.r[q] - s;
  } else if (MODE == R_JAC) {
    ep.y[q] = x[q] + (ep.r[q] - s) / ep.d[i];
  } else {
    const double d = ep.d[i];
    double f = d != 0. ? ep.c2 * (ep.r[q] - s) / d : 0.;
    if (ep.c1 != 0.) f += ep.c1 * ep.dd[q];
    ep.dd[q] = f;
    ep.y[q] = x[q] + f;
  }
}

template <int K>
__device__ __forceinline__ void r_load(const double *__restrict__ p, double (&v)[K]) {
  if constexpr (K == 1) {
    v[0] = p[0];
  } else {
#pragma unroll
    for (int h = 0; h < K / 2; ++h) {
      const double2 t = reinterpret_cast<const double2 *>(p)[h];
      v[2 * h] = t.x;
      v[2 * h + 1] = t.y;
    }
  }
}

// Sums the K columns over W lanes: each exchange halves the columns a lane
// carries until it carries one (col), then halves the lanes.  Lanes whose
// low W / K bits are zero hold column col's sum.
template <int K, int W>
__device__ __forceinline__ double r_reduce(const double (&a)[K], int lane, int &col) {
  if constexpr (W == 1) {
    return a[0];
  } else if constexpr (K == 1) {
    const double b[1] = {a[0] + __shfl_xor(a[0], W / 2)};
    return r_reduce<1, W / 2>(b, lane, col);
  } else {
    constexpr int H = K / 2;
    const bool up = (lane & (W / 2)) != 0;
    double b[H];
#pragma unroll
    for (int q = 0; q < H; ++q) {
      const double keep = up ? a[H + q] : a[q], send = up ? a[q] : a[H + q];
      b[q] = keep + __shfl_xor(send, W / 2);
    }
    if (up) col += H;
    return r_reduce<H, W / 2>(b, lane, col);
  }
}

// The first nbw workgroups give every chunk of a listed row (kLongRow) a
// wavefront, a lane per entry and K columns a lane; rows of several chunks
// leave partial sums to k_rm_fin.  The rest take the short rows, 8 lanes each.
// One workgroup per row above 64 entries, in a launch of its own (the layout
// before), took 28 us a product at 200x200x24, whose longest rows hold 1e5
// entries, and served one column.
template <int K, int MODE>
__global__ void __launch_bounds__(256) k_rm(int64_t nr, unsigned nbw, const int64_t *__restrict__ rp,
                                            const int32_t *__restrict__ ci, const double *__restrict__ v,
                                            const int32_t *__restrict__ lidx, const int32_t *__restrict__ lrows,
                                            const int64_t *__restrict__ lcb, const int64_t *__restrict__ lce, int nchunk,
                                            int nsingle, const double *x, REp ep, double *__restrict__ part) {
  double a[K];
#pragma unroll
  for (int q = 0; q < K; ++q) a[q] = 0.;
  if (blockIdx.x < nbw) {
    const int c = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (c >= nchunk) return;  // uniform across the wavefront
    const int lane = threadIdx.x & 63;
    const int64_t b = lcb[c], e = lce[c];
    constexpr int NB = (int)(kLongChunk / 64);
    int32_t cc[NB];
    double av[NB];
#pragma unroll
    for (int h = 0; h < NB; ++h) {  // past the end: the last entry's column with value 0
      const int64_t p = b + h * 64 + lane, pp = p < e ? p : e - 1;
      cc[h] = ci[pp];
      av[h] = p < e ? v[pp] : 0.;
    }
#pragma unroll
    for (int h = 0; h < NB; ++h) {
      if (b + h * 64 >= e) break;
      double xv[K];
      r_load<K>(x + (int64_t)cc[h] * K, xv);
#pragma unroll
      for (int q = 0; q < K; ++q) a[q] += av[h] * xv[q];
    }
    int col = 0;
    const double s = r_reduce<K, 64>(a, lane, col);
    if (lane & (64 / K - 1)) return;
    if (c < nsingle) r_row<K, MODE>(ep, x, lrows[c], col, s);
    else part[(int64_t)(c - nsingle) * K + col] = s;
    return;
  }
  const int64_t i = ((int64_t)(blockIdx.x - nbw) * 256 + threadIdx.x) >> 3;
  const int lane = threadIdx.x & 7;
  if (i >= nr || (lidx && lidx[i] >= 0)) return;  // the same on a row's 8 lanes
  const int64_t b = rp[i], e = rp[i + 1];
  constexpr int NB = (int)(kLongRow / 8);
  int32_t cc[NB];
  double av[NB];
#pragma unroll
  for (int h = 0; h < NB; ++h) {
    const int64_t p = b + h * 8 + lane;
    cc[h] = 0;
    av[h] = 0.;
    if (p < e) { cc[h] = ci[p]; av[h] = v[p]; }
  }
#pragma unroll
  for (int h = 0; h < NB; ++h)
    if (b + h * 8 + lane < e) {
      double xv[K];
      r_load<K>(x + (int64_t)cc[h] * K, xv);
#pragma unroll
      for (int q = 0; q < K; ++q) a[q] += av[h] * xv[q];
    }
  int col = 0;
  const double s = r_reduce<K, 8>(a, lane, col);
  if ((lane & (8 / K - 1)) == 0) r_row<K, MODE>(ep, x, i, col, s);
}
static_assert(kLongRow % 8 == 0 && kLongChunk % 64 == 0, "rounds of the row walks");

// rows of several chunks: a wavefront per row sums the partial sums
template <int K, int MODE>
__global__ void __launch_bounds__(256) k_rm_fin(int nmulti, int nsingle, const int32_t *__restrict__ lrows,
                                                const int32_t *__restrict__ lqp, const double *x, REp ep,
                                                const double *__restrict__ part) {
  const int r = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if (r >= nmulti) return;  // uniform across the wavefront
  const int lane = threadIdx.x & 63;
  double a[K];
#pragma unroll
  for (int q = 0; q < K; ++q) a[q] = 0.;
  for (int c = lqp[nsingle + r] + lane; c < lqp[nsingle + r + 1]; c += 64) {
    double t[K];
    r_load<K>(part + (int64_t)(c - nsingle) * K, t);
#pragma unroll
    for (int q = 0; q < K; ++q) a[q] += t[q];
  }
  int col = 0;
  const double s = r_reduce<K, 64>(a, lane, col);
  if ((lane & (64 / K - 1)) == 0) r_row<K, MODE>(ep, x, lrows[nsingle + r], col, s);
}

// x = inv r on the coarsest level, one wavefront per row (coalesced rows)
template <int K>
__global__ void k_r_dense(int64_t n, const double *__restrict__ inv, const double *__restrict__ r, double *__restrict__ x) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64;
  const int lane = threadIdx.x & 63;
  if (i >= n) return;
  double a[K];
#pragma unroll
  for (int q = 0; q < K; ++q) a[q] = 0.;
#pragma unroll 4
  for (int64_t j = lane; j < n; j += 64) {
    const double m = inv[i * n + j];
    double t[K];
    r_load<K>(r + j * K, t);
#pragma unroll
    for (int q = 0; q < K; ++q) a[q] += m * t[q];
  }
  int col = 0;
  const double s = r_reduce<K, 64>(a, lane, col);
  if ((lane & (64 / K - 1)) == 0) x[i * K + col] = s;
}

// ---------------------------------------------------------------- Krylov kernels of K columns

// partial[(blk * nvec + t) * K + j] = sum over the block's rows of V_t w, four
// vectors per grid row
constexpr int kRDotBlocks = 256, kRDotChunk = 4;
template <int K>
__global__ void __launch_bounds__(256) k_rm_dots(int64_t n, const double *__restrict__ V, int64_t vstride, int nvec,
                                                 const double *__restrict__ w, double *__restrict__ partial) {
  __shared__ double sh[256];
  const int t0 = blockIdx.y * kRDotChunk, nt = min(kRDotChunk, nvec - t0);
  double acc[kRDotChunk] = {0., 0., 0., 0.};
  for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < n * K; q += (int64_t)gridDim.x * 256) {  // 256 % K == 0
    const double b = w[q];
#pragma unroll
    for (int t = 0; t < kRDotChunk; ++t)
      if (t < nt) acc[t] += V[(int64_t)(t0 + t) * vstride + q] * b;
  }
  for (int t = 0; t < nt; ++t) {
    sh[threadIdx.x] = acc[t];
    __syncthreads();
    for (int h = 128; h >= K; h >>= 1) {
      if ((int)threadIdx.x < h) sh[threadIdx.x] += sh[threadIdx.x + h];
      __syncthreads();
    }
    if ((int)threadIdx.x < K) partial[((int64_t)blockIdx.x * nvec + t0 + t) * K + threadIdx.x] = sh[threadIdx.x];
    __syncthreads();
  }
}

// h[q] = the sum of the blocks' partial sums of output q, a wavefront each
__global__ void k_rm_dots_fin(int nout, int nb, const double *__restrict__ partial, double *__restrict__ h) {
  const int q = (int)(blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64), lane = threadIdx.x & 63;
  if (q >= nout) return;  // uniform across the wavefront
  double a = 0.;
  for (int b = lane; b < nb; b += 64) a += partial[(int64_t)b * nout + q];
  for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o);
  if (lane == 0) h[q] = a;
}

// w -= sum_t V_t h_t
template <int K>
__global__ void k_rm_gs(int64_t n, const double *__restrict__ V, int64_t vstride, int nvec, const double *__restrict__ h,
                        double *__restrict__ w) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n * K) return;
  const int j = (int)(q % K);
  double a = w[q];
#pragma unroll 4
  for (int t = 0; t < nvec; ++t) a -= V[(int64_t)t * vstride + q] * h[t * K + j];
  w[q] = a;
}

// w *= sc_j, or (sc null) divided by sqrt(nn_j) where that is positive; with z
// also the finest level's first sweep from zero, z = dd = zc w / d
template <int K>
__global__ void k_rm_scale(int64_t n, const double *__restrict__ sc, const double *__restrict__ nn,
                           double *__restrict__ w, const double *__restrict__ d, double zc, double *__restrict__ z,
                           double *__restrict__ dd) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n * K) return;
  const int j = (int)(q % K);
  const double f = sc ? sc[j] : nn[j] > 0. ? 1.0 / sqrt(nn[j]) : 1.0;
  const double v = w[q] * f;
  w[q] = v;
  if (!z) return;
  const double di = d[q / K], g = di != 0. ? zc * v / di : 0.;
  z[q] = g;
  if (dd) dd[q] = g;
}

// x += sum_t Z_t y_t
template <int K>
__global__ void k_rm_xup(int64_t n, const double *__restrict__ Z, int64_t zstride, int nvec, const double *__restrict__ y,
                         double *__restrict__ x) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n * K) return;
  const int j = (int)(q % K);
  double a = x[q];
#pragma unroll 4
  for (int t = 0; t < nvec; ++t) a += Z[(int64_t)t * zstride + q] * y[t * K + j];
  x[q] = a;
}

__global__ void k_csr_dense(int64_t n, int64_t nnz, const int64_t *__restrict__ rp, const int32_t *__restrict__ ci,
                            const double *__restrict__ v, double *__restrict__ out) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p < nnz) out[csr_row_of(rp, n, p) * n + ci[p]] = v[p];  // columns of a row are distinct
}

}  // namespace

struct RLevel {
  Csr A, P, R;              // rows above kLongRow listed
  double *d = nullptr, *dl1 = nullptr;
  double c1[kChebSteps] = {}, c2[kChebSteps] = {};  // Chebyshev coefficients of each step
};

constexpr int kRestart = 30;

// Vectors of a solve of K columns, kept for the next one of as many or fewer.
struct RWork {
  int K = 0;
  Arena A;
  std::vector<double *> r, x, t, dd;  // per level (r: from level 1 on)
  double *part = nullptr;             // partial sums of the longest rows
  // FGMRES: basis V (m+1 vectors), preconditioned basis Z (m), partial sums of
  // the dot products, their results, per-column factors
  double *V = nullptr, *Zb = nullptr, *dpart = nullptr, *h = nullptr, *y = nullptr;
};

struct RealAMG {
  int smoother = GP_SMOOTH_L1_JACOBI;
  std::vector<RLevel> L;
  double *inv = nullptr;  // coarsest, dense n x n
  Arena A;
  RWork W;
};

namespace {

// the Chebyshev coefficients for lambda, the estimate of D^-1 A's largest
// eigenvalue: interval [alpha, beta], theta its centre, delta its half width,
// sigma = theta / delta; step 0: c1 = 0, c2 = 1 / theta; step k: rho_k =
// 1 / (2 sigma - rho_(k-1)) from rho_0 = 1 / sigma, c1 = rho_k rho_(k-1),
// c2 = 2 rho_k / delta
void cheb_coeffs(double lam, double *c1, double *c2) {
  const double beta = kChebUpper * lam, alpha = kChebLower * beta;
  const double theta = 0.5 * (beta + alpha), delta = 0.5 * (beta - alpha), sigma = theta / delta;
  double rho = 1.0 / sigma;
  c1[0] = 0.;
  c2[0] = 1.0 / theta;
  for (int k = 1; k < kChebSteps; ++k) {
    const double rn = 1.0 / (2.0 * sigma - rho);
    c1[k] = rn * rho;
    c2[k] = 2.0 * rn / delta;
    rho = rn;
  }
}

// one pairwise matching pass on M: tentative P (n x ncoarse)
gp_status match_pass(Arena &A, Arena &tmp, const Csr &M, const double *d, Csr *P, hipStream_t s) {
  const int64_t n = M.nr;
  int32_t *matched, *mnext, *pick, *partner;
  int64_t *root, *rscan;
  GP_TRY(tmp.alloc(&matched, n)); GP_TRY(tmp.alloc(&mnext, n)); GP_TRY(tmp.alloc(&pick, n));
  GP_TRY(tmp.alloc(&partner, n)); GP_TRY(tmp.alloc(&root, n)); GP_TRY(tmp.alloc(&rscan, n + 1));
  GP_HIP(hipMemsetAsync(matched, 0, sizeof(int32_t) * n, s));
  GP_HIP(hipMemsetAsync(mnext, 0, sizeof(int32_t) * n, s));
  GP_HIP(hipMemsetAsync(partner, 0xff, sizeof(int32_t) * n, s));  // -1
  for (int round = 0; round < 6; ++round) {
    k_pick<<<wave_blocks(n), 256, 0, s>>>(n, M.rp, M.ci, M.v[0], d, matched, pick);
    k_pair<<<blocks_for(n), 256, 0, s>>>(n, pick, partner, mnext);
    k_copy_i32<<<blocks_for(n), 256, 0, s>>>(n, mnext, matched);
  }
  k_roots<<<blocks_for(n), 256, 0, s>>>(n, partner, root);
  GP_TRY(exclusive_scan_i64(root, rscan, n, s, tmp));
  int64_t nc = 0;
  GP_HIP(hipMemcpyAsync(&nc, rscan + n, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  GP_HIP(hipStreamSynchronize(s));
  GP_TRY(csr_alloc(A, n, nc, n, 1, P));
  k_ptent_pairs<<<blocks_for(n + 1), 256, 0, s>>>(n, partner, rscan, P->rp, P->ci, P->v[0]);
  GP_HIP(hipStreamSynchronize(s));
  return GP_OK;
}

__global__ void k_r_fill_hash(int64_t n, double *__restrict__ x) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = 0.5 + 0.5 * (double)((i * 2654435761ULL) % 1000) / 1000.0;
}

// largest eigenvalue of D^-1 A by 12 power iterations, the norms kept on the
// device (vectors went to the host and back at each before: 24 copies of n)
gp_status power_lambda(Arena &tmp, const Csr &M, const double *d, double *lam, hipStream_t s) {
  const int64_t n = M.nr;
  double *x, *y, *part, *nrm;
  GP_TRY(tmp.alloc(&x, n)); GP_TRY(tmp.alloc(&y, n)); GP_TRY(tmp.alloc(&part, kNormBlocks)); GP_TRY(tmp.alloc(&nrm, 1));
  k_r_fill_hash<<<blocks_for(n), 256, 0, s>>>(n, x);
  for (int it = 0; it < 12; ++it) {
    k_r_dinv_spmv<<<wave_blocks(n), 256, 0, s>>>(n, M.rp, M.ci, M.v[0], d, x, y);
    GP_TRY(dev_norm(y, n, part, nrm, s));  // |D^-1 A x| with |x| = 1 after the first step
    GP_TRY(dev_div(y, n, nrm, s));
    std::swap(x, y);
  }
  double h = 0.;
  GP_HIP(hipMemcpyAsync(&h, nrm, sizeof(double), hipMemcpyDeviceToHost, s));
  GP_HIP(hipStreamSynchronize(s));
  *lam = std::max(h, 1e-3);
  return GP_OK;
}

gp_status build_real_amg(RealAMG &G, Csr A0, hipStream_t s) {
  Arena &A = G.A;
  G.L.clear();
  RLevel l0;
  l0.A = A0;
  G.L.push_back(l0);
  for (;;) {
    RLevel &F = G.L.back();
    const int64_t n = F.A.nr;
    GP_TRY(A.alloc(&F.d, n)); GP_TRY(A.alloc(&F.dl1, n));
    k_r_diag<<<wave_blocks(n), 256, 0, s>>>(n, F.A.rp, F.A.ci, F.A.v[0], F.d, F.dl1);
    GP_TRY(csr_mark_long(A, F.A, s));
    if (n <= kCoarsest || G.L.size() >= 24) break;
    TmpArena tmp;
    gp_status st = GP_OK;
    Csr P1, M2, AP1, P2, Pt, DA, DAP, Ps, P, AP, Ac, R;
    do {
      if ((st = match_pass(tmp, tmp, F.A, F.d, &P1, s)) != GP_OK) break;
      Csr R1;
      if ((st = transpose(tmp, P1, &R1, s)) != GP_OK) break;
      if ((st = spgemm(tmp, F.A, P1, &AP1, s)) != GP_OK) break;
      if ((st = spgemm(tmp, R1, AP1, &M2, s)) != GP_OK) break;
      double *d2 = nullptr, *l2 = nullptr;
      if ((st = tmp.alloc(&d2, M2.nr)) != GP_OK || (st = tmp.alloc(&l2, M2.nr)) != GP_OK) break;
      k_r_diag<<<wave_blocks(M2.nr), 256, 0, s>>>(M2.nr, M2.rp, M2.ci, M2.v[0], d2, l2);
      if ((st = match_pass(tmp, tmp, M2, d2, &P2, s)) != GP_OK) break;
      if ((st = spgemm(tmp, P1, P2, &Pt, s)) != GP_OK) break;
      if (Pt.nc > (int64_t)(0.8 * (double)n)) { st = GP_ERR_NOCONV; break; }  // stalled: stop coarsening
      // P = Pt - 4/(3 lambda) D^-1 A Pt
      double lam = 2.0;
      if ((st = power_lambda(tmp, F.A, F.d, &lam, s)) != GP_OK) break;
      if (G.smoother == GP_SMOOTH_CHEBYSHEV) cheb_coeffs(lam, F.c1, F.c2);
      if ((st = csr_alloc(tmp, n, n, F.A.nnz, 1, &DA)) != GP_OK) break;
      if (hipMemcpyAsync(DA.rp, F.A.rp, sizeof(int64_t) * (n + 1), hipMemcpyDeviceToDevice, s) != hipSuccess ||
          hipMemcpyAsync(DA.ci, F.A.ci, sizeof(int32_t) * F.A.nnz, hipMemcpyDeviceToDevice, s) != hipSuccess) { st = fail(GP_ERR_HIP, "copy"); break; }
      k_r_scale_rows<<<blocks_for(F.A.nnz), 256, 0, s>>>(n, F.A.nnz, F.A.rp, F.A.v[0], F.d, 4.0 / (3.0 * lam), DA.v[0]);
      if ((st = spgemm(tmp, DA, Pt, &DAP, s)) != GP_OK) break;
      if ((st = csr_add(tmp, Pt, -1.0, DAP, &Ps, s)) != GP_OK) break;
      if ((st = truncate_prolongation(A, tmp, Ps, Pt, kTrunc, &P, s)) != GP_OK) break;
      if ((st = transpose(A, P, &R, s)) != GP_OK) break;
      if ((st = spgemm(tmp, F.A, P, &AP, s)) != GP_OK) break;
      if ((st = spgemm(A, R, AP, &Ac, s)) != GP_OK) break;
    } while (0);
    tmp.free_all();
    if (st == GP_ERR_NOCONV) { (void)hipGetLastError(); break; }
    if (st != GP_OK) return st;
    F.P = P;
    F.R = R;
    GP_TRY(csr_mark_long(A, F.P, s));
    GP_TRY(csr_mark_long(A, F.R, s));
    RLevel C;
    C.A = Ac;
    G.L.push_back(C);
  }
  // coarsest: dense inverse on the device
  RLevel &C = G.L.back();
  const int64_t n = C.A.nr;
  if (n > 4096) return fail(GP_ERR_NOCONV, "real AMG coarsening stalled above 4096 unknowns");
  GP_TRY(A.alloc(&G.inv, std::max<int64_t>(n * n, 1)));
  GP_HIP(hipMemsetAsync(G.inv, 0, sizeof(double) * n * n, s));
  if (C.A.nnz) k_csr_dense<<<blocks_for(C.A.nnz), 256, 0, s>>>(n, C.A.nnz, C.A.rp, C.A.ci, C.A.v[0], G.inv);
  GP_TRY(dense_inverse_real(G.inv, (int)n, s));
  GP_HIP(hipStreamSynchronize(s));
  return GP_OK;
}

template <int K, int MODE>
void rm(const Csr &M, const double *v, const double *x, const REp &ep, double *part, hipStream_t s) {
  if (M.nr == 0) return;
  const unsigned nbw = (unsigned)((M.nchunk + 3) / 4);
  const unsigned nbs = M.nlong == M.nr ? 0u : (unsigned)((M.nr * 8 + 255) / 256);
  k_rm<K, MODE><<<nbw + nbs, 256, 0, s>>>(M.nr, nbw, M.rp, M.ci, v, M.lidx, M.lrows, M.lcb, M.lce, M.nchunk, M.nsingle, x,
                                          ep, part);
  const int nmulti = M.nlong - M.nsingle;
  if (nmulti)
    k_rm_fin<K, MODE><<<(unsigned)((nmulti + 3) / 4), 256, 0, s>>>(nmulti, M.nsingle, M.lrows, M.lqp, x, ep, part);
}

template <int K>
struct RCycle {
  const RealAMG &G;
  RWork &W;
  hipStream_t s;
  bool cheb() const { return G.smoother == GP_SMOOTH_CHEBYSHEV; }
  double first_c(int l) const { return cheb() ? G.L[l].c2[0] : 1.0; }
  const double *first_d(int l) const { return cheb() ? G.L[l].d : G.L[l].dl1; }
  // step k of the smoother (k = 0: from a nonzero x)
  void smooth(int l, int k, const double *r, const double *x, double *y) {
    const RLevel &L = G.L[l];
    REp ep;
    ep.r = r; ep.y = y;
    if (cheb()) {
      ep.d = L.d; ep.c1 = L.c1[k]; ep.c2 = L.c2[k]; ep.dd = W.dd[l];
      rm<K, R_CHEB>(L.A, L.A.v[0], x, ep, W.part, s);
    } else {
      ep.d = L.dl1;
      rm<K, R_JAC>(L.A, L.A.v[0], x, ep, W.part, s);
    }
  }
  // One V-cycle on level l for the right-hand side r, whose first sweep from
  // zero is in W.x[l] (and W.dd[l]) already; the result goes to out.
  void run(int l, const double *r, double *out) {
    const RLevel &L = G.L[l];
    if (l + 1 == (int)G.L.size()) {
      k_r_dense<K><<<blocks_for(L.A.nr * 64), 256, 0, s>>>(L.A.nr, G.inv, r, out);
      return;
    }
    static_assert(kChebSteps == 2, "the smoothing steps alternate between x and t twice");
    double *x = W.x[l], *t = W.t[l];
    smooth(l, 1, r, x, t);
    REp res;
    res.r = r; res.y = x;                       // x <- r - A t
    rm<K, R_RES>(L.A, L.A.v[0], t, res, W.part, s);
    REp down;
    down.y = W.r[l + 1];
    if (l + 2 < (int)G.L.size()) {
      down.z = W.x[l + 1]; down.zd = first_d(l + 1); down.zc = first_c(l + 1);
      if (cheb()) down.dd = W.dd[l + 1];
    }
    rm<K, R_MUL>(L.R, L.R.v[0], x, down, W.part, s);
    run(l + 1, W.r[l + 1], W.t[l + 1]);
    REp up;
    up.y = t; up.acc = 1;                       // t += P xc
    rm<K, R_MUL>(L.P, L.P.v[0], W.t[l + 1], up, W.part, s);
    smooth(l, 0, r, t, x);
    smooth(l, 1, r, x, out);
  }
};

gp_status work(RealAMG &G, int K) {
  RWork &W = G.W;
  if (W.K >= K) return GP_OK;
  W.A.free_all();
  W.K = 0;
  const size_t nl = G.L.size();
  const int64_t n = G.L[0].A.nr;
  W.r.assign(nl, nullptr); W.x.assign(nl, nullptr); W.t.assign(nl, nullptr); W.dd.assign(nl, nullptr);
  int64_t chunks = 0;
  for (size_t l = 0; l < nl; ++l) {
    const RLevel &L = G.L[l];
    if (l) GP_TRY(W.A.alloc(&W.r[l], L.A.nr * K));
    GP_TRY(W.A.alloc(&W.x[l], L.A.nr * K)); GP_TRY(W.A.alloc(&W.t[l], L.A.nr * K));
    if (G.smoother == GP_SMOOTH_CHEBYSHEV) GP_TRY(W.A.alloc(&W.dd[l], L.A.nr * K));
    for (const Csr *M : {&L.A, &L.P, &L.R}) chunks = std::max<int64_t>(chunks, M->nchunk);
  }
  GP_TRY(W.A.alloc(&W.part, std::max<int64_t>(chunks, 1) * K));
  GP_TRY(W.A.alloc(&W.V, (int64_t)(kRestart + 1) * n * K));
  GP_TRY(W.A.alloc(&W.Zb, (int64_t)kRestart * n * K));
  GP_TRY(W.A.alloc(&W.dpart, (int64_t)kRDotBlocks * (kRestart + 1) * K));
  GP_TRY(W.A.alloc(&W.h, (int64_t)(2 * kRestart + 1) * K));
  GP_TRY(W.A.alloc(&W.y, (int64_t)kRestart * K));
  W.K = K;
  return GP_OK;
}

template <int K>
void rdots(const RWork &W, int64_t n, const double *V, int nvec, const double *w, double *h, hipStream_t s) {
  k_rm_dots<K><<<dim3(kRDotBlocks, (nvec + kRDotChunk - 1) / kRDotChunk), 256, 0, s>>>(n, V, n * K, nvec, w, W.dpart);
  k_rm_dots_fin<<<(unsigned)((nvec * K + 3) / 4), 256, 0, s>>>(nvec * K, kRDotBlocks, W.dpart, h);
}

// Flexible GMRES(m) per column, FP64, classical Gram-Schmidt with one
// reorthogonalization pass, Givens rotations on the host: the coefficients of
// both passes and the norm stay on the device and reach the host once per step.
template <int K>
gp_status solve_cols(RealAMG &G, const double *bd, double *xd, double tol, int maxit, int32_t *iters, double *relres,
                     hipStream_t s) {
  const int m = kRestart;
  RWork &W = G.W;
  const RLevel &L0 = G.L[0];
  const int64_t n = L0.A.nr, nk = n * K;
  RCycle<K> cyc{G, W, s};
  const bool one = G.L.size() == 1;
  const unsigned gk = blocks_for(nk);
  GP_HIP(hipMemsetAsync(xd, 0, sizeof(double) * nk, s));
  std::vector<double> hh((size_t)(2 * m + 1) * K);
  auto fetch = [&](const double *dv, int cnt) -> gp_status {
    GP_HIP(hipMemcpyAsync(hh.data(), dv, sizeof(double) * cnt, hipMemcpyDeviceToHost, s));
    GP_HIP(hipStreamSynchronize(s));
    return GP_OK;
  };
  rdots<K>(W, n, bd, 1, bd, W.h, s);
  GP_TRY(fetch(W.h, K));
  double bn[K], rel[K], beta[K], sc[K];
  bool active[K];
  for (int j = 0; j < K; ++j) { bn[j] = std::sqrt(hh[j]); rel[j] = 0.; iters[j] = 0; }
  std::vector<double> H((size_t)(m + 1) * m * K), cs((size_t)m * K), sn((size_t)m * K), g((size_t)(m + 1) * K),
      y((size_t)m * K);
  for (;;) {
    REp res;
    res.r = bd; res.y = W.V;
    rm<K, R_RES>(L0.A, L0.A.v[0], xd, res, W.part, s);
    rdots<K>(W, n, W.V, 1, W.V, W.h, s);
    GP_TRY(fetch(W.h, K));
    bool any = false;
    for (int j = 0; j < K; ++j) {
      beta[j] = std::sqrt(hh[j]);
      active[j] = false;
      if (bn[j] > 0.) {
        rel[j] = beta[j] / bn[j];
        active[j] = rel[j] > tol && iters[j] < maxit;
      }
      sc[j] = active[j] ? 1.0 / beta[j] : 0.;
      any = any || active[j];
    }
    if (!any) break;
    // columns that are done carry zero vectors
    GP_HIP(hipMemcpyAsync(W.y, sc, sizeof(double) * K, hipMemcpyHostToDevice, s));
    auto scale = [&](const double *scp, double *v) {
      k_rm_scale<K><<<gk, 256, 0, s>>>(n, scp, W.h + (int64_t)2 * m * K, v, cyc.first_d(0), cyc.first_c(0),
                                       one ? nullptr : W.x[0], W.dd[0]);
    };
    scale(W.y, W.V);
    std::fill(g.begin(), g.end(), 0.);
    for (int j = 0; j < K; ++j) g[j] = active[j] ? beta[j] : 0.;
    int used[K] = {}, steps = 0;
    bool open[K];
    for (int j = 0; j < K; ++j) open[j] = active[j];
    for (int i = 0; i < m; ++i) {
      double *Vi = W.V + (int64_t)i * nk, *Vn = Vi + nk, *Zi = W.Zb + (int64_t)i * nk;
      cyc.run(0, Vi, Zi);
      REp mul;
      mul.y = Vn;
      rm<K, R_MUL>(L0.A, L0.A.v[0], Zi, mul, W.part, s);
      double *h1 = W.h, *h2 = W.h + (int64_t)(i + 1) * K, *nn = W.h + (int64_t)2 * m * K;
      for (double *h : {h1, h2}) {
        rdots<K>(W, n, W.V, i + 1, Vn, h, s);
        k_rm_gs<K><<<gk, 256, 0, s>>>(n, W.V, nk, i + 1, h, Vn);
      }
      rdots<K>(W, n, Vn, 1, Vn, nn, s);
      scale(nullptr, Vn);
      GP_TRY(fetch(W.h, (2 * m + 1) * K));
      steps = i + 1;
      bool more = false;
      for (int j = 0; j < K; ++j) {
        if (!open[j]) continue;
        double *Hj = &H[(size_t)j * (m + 1) * m], *cj = &cs[(size_t)j * m], *sj = &sn[(size_t)j * m];
        for (int t = 0; t <= i; ++t) Hj[t * m + i] = hh[t * K + j] + hh[(i + 1 + t) * K + j];
        Hj[(i + 1) * m + i] = std::sqrt(std::max(hh[(size_t)2 * m * K + j], 0.));
        for (int t = 0; t < i; ++t) {
          const double a = Hj[t * m + i], bq = Hj[(t + 1) * m + i];
          Hj[t * m + i] = cj[t] * a + sj[t] * bq;
          Hj[(t + 1) * m + i] = -sj[t] * a + cj[t] * bq;
        }
        const double a = Hj[i * m + i], bq = Hj[(i + 1) * m + i];
        const double den = std::sqrt(a * a + bq * bq);
        cj[i] = den > 0 ? a / den : 1.;
        sj[i] = den > 0 ? bq / den : 0.;
        Hj[i * m + i] = cj[i] * a + sj[i] * bq;
        Hj[(i + 1) * m + i] = 0.;
        g[(i + 1) * K + j] = -sj[i] * g[i * K + j];
        g[i * K + j] = cj[i] * g[i * K + j];
        ++iters[j];
        used[j] = i + 1;
        if (std::fabs(g[(i + 1) * K + j]) <= tol * bn[j] || iters[j] >= maxit) open[j] = false;
        more = more || open[j];
      }
      if (!more) break;
    }
    std::fill(y.begin(), y.end(), 0.);
    for (int j = 0; j < K; ++j) {
      const double *Hj = &H[(size_t)j * (m + 1) * m];
      for (int t = used[j] - 1; t >= 0; --t) {
        double acc = g[t * K + j];
        for (int q = t + 1; q < used[j]; ++q) acc -= Hj[t * m + q] * y[q * K + j];
        y[t * K + j] = Hj[t * m + t] != 0. ? acc / Hj[t * m + t] : 0.;
      }
    }
    GP_HIP(hipMemcpyAsync(W.y, y.data(), sizeof(double) * steps * K, hipMemcpyHostToDevice, s));
    k_rm_xup<K><<<gk, 256, 0, s>>>(n, W.Zb, nk, steps, W.y, xd);
  }
  GP_HIP(hipStreamSynchronize(s));
  GP_HIP(hipGetLastError());
  bool ok = true;
  for (int j = 0; j < K; ++j) { relres[j] = rel[j]; ok = ok && rel[j] <= tol; }
  return ok ? GP_OK : fail(GP_ERR_NOCONV, "real solve stopped above the tolerance");
}

}  // namespace

gp_status real_amg_create(int64_t n, int64_t nnz, const int64_t *rows, const int64_t *cols, const double *vals,
                          int smoother, RealAMG **out, hipStream_t s) {
  *out = nullptr;
  if (n < 1 || nnz < 1) return fail(GP_ERR_ARG, "empty real matrix");
  if (n > 2147483647LL) return fail(GP_ERR_ARG, "more than 2^31 unknowns");
  if (smoother != GP_SMOOTH_L1_JACOBI && smoother != GP_SMOOTH_CHEBYSHEV) return fail(GP_ERR_ARG, "unknown real smoother");
  RealAMG *G = new RealAMG();
  G->smoother = smoother;
  Csr A0;
  const double *vv[1] = {vals};
  gp_status st = csr_from_coo(G->A, n, n, nnz, rows, cols, vv, 1, &A0, s);
  if (st == GP_OK) st = build_real_amg(*G, A0, s);
  if (st != GP_OK) { real_amg_destroy(G); return st; }
  *out = G;
  return GP_OK;
}

int64_t real_amg_rows(const RealAMG *G) { return G->L[0].A.nr; }
int32_t real_amg_levels(const RealAMG *G) { return (int32_t)G->L.size(); }
int64_t real_amg_column_bytes(const RealAMG *G) {
  int64_t rows = (2 * kRestart + 1) * G->L[0].A.nr;
  for (const RLevel &L : G->L) rows += 4 * L.A.nr;
  return (int64_t)sizeof(double) * rows;
}
int64_t real_amg_work_bytes(const RealAMG *G) { return G->W.A.bytes; }
int64_t real_amg_bytes(const RealAMG *G) { return G->A.bytes + G->W.A.bytes; }

void real_amg_trim(RealAMG *G) {
  if (!G) return;
  G->W.A.free_all();
  G->W.K = 0;
}

void real_amg_destroy(RealAMG *G) {
  if (!G) return;
  G->W.A.free_all();
  G->A.free_all();
  delete G;
}

gp_status real_amg_solve(RealAMG *G, int k, const double *b, double *x, double tol, int maxit, int32_t *iters,
                         double *relres, hipStream_t s) {
  if (k != 1 && k != 2 && k != 4 && k != 8) return fail(GP_ERR_ARG, "real solves take 1, 2, 4 or 8 columns");
  GP_TRY(work(*G, k));
  if (k == 1) return solve_cols<1>(*G, b, x, tol, maxit, iters, relres, s);
  if (k == 2) return solve_cols<2>(*G, b, x, tol, maxit, iters, relres, s);
  if (k == 4) return solve_cols<4>(*G, b, x, tol, maxit, iters, relres, s);
  return solve_cols<8>(*G, b, x, tol, maxit, iters, relres, s);
}

gp_status real_mv(const Csr &M, int which, int k, double alpha, int acc, const double *x, double *y, double *part,
                  hipStream_t s) {
  REp ep;
  ep.y = y; ep.alpha = alpha; ep.acc = acc;
  if (k == 1) rm<1, R_MUL>(M, M.v[which], x, ep, part, s);
  else if (k == 2) rm<2, R_MUL>(M, M.v[which], x, ep, part, s);
  else if (k == 4) rm<4, R_MUL>(M, M.v[which], x, ep, part, s);
  else if (k == 8) rm<8, R_MUL>(M, M.v[which], x, ep, part, s);
  else return fail(GP_ERR_ARG, "real products take 1, 2, 4 or 8 columns");
  GP_HIP(hipGetLastError());
  return GP_OK;
}

}  // namespace gp

using namespace gp;

extern "C" gp_status gp_solve_real(const int64_t *row, const int64_t *col, const double *val, int64_t nnz, int64_t n,
                                   const double *b, double *x, double rtol, int32_t *iters_out, double *relres_out) {
  return gp_solve_real_ex(row, col, val, nnz, n, b, x, rtol, GP_SMOOTH_L1_JACOBI, iters_out, relres_out);
}

extern "C" gp_status gp_solve_real_ex(const int64_t *row, const int64_t *col, const double *val, int64_t nnz,
                                      int64_t n, const double *b, double *x, double rtol, int32_t smoother,
                                      int32_t *iters_out, double *relres_out) {
  if (!row || !col || !val || !b || !x || n < 1 || nnz < 1) return fail(GP_ERR_ARG, "bad real solve arguments");
  if (smoother != GP_SMOOTH_L1_JACOBI && smoother != GP_SMOOTH_CHEBYSHEV) return fail(GP_ERR_ARG, "unknown real smoother");
  if (n > 2147483647LL) return fail(GP_ERR_ARG, "more than 2^31 unknowns");
  for (int64_t q = 0; q < nnz; ++q)
    if (row[q] < 0 || row[q] >= n || col[q] < 0 || col[q] >= n) return fail(GP_ERR_ARG, "COO index out of range");
  GP_TRY(ensure_device());
  const double tol = rtol > 0 ? rtol : 1e-4;  // the reference's HYPRE tolerance (src/hypreSolver.h:8)
  hipStream_t s;
  GP_HIP(hipStreamCreate(&s));
  struct StreamGuard { hipStream_t s; ~StreamGuard() { (void)hipStreamSynchronize(s); (void)hipStreamDestroy(s); } } sg{s};
  ScratchScope scratch(s);
  TmpArena tmp;
  struct TGuard { Arena *a; hipStream_t s; ~TGuard() { (void)hipStreamSynchronize(s); a->free_all(); } } tg{&tmp, s};
  int64_t *dr, *dc;
  double *dv, *bd, *xd;
  GP_TRY(tmp.alloc(&dr, nnz)); GP_TRY(tmp.alloc(&dc, nnz)); GP_TRY(tmp.alloc(&dv, nnz));
  GP_TRY(tmp.alloc(&bd, n)); GP_TRY(tmp.alloc(&xd, n));
  GP_HIP(hipMemcpyAsync(dr, row, sizeof(int64_t) * nnz, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(dc, col, sizeof(int64_t) * nnz, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(dv, val, sizeof(double) * nnz, hipMemcpyHostToDevice, s));
  GP_HIP(hipMemcpyAsync(bd, b, sizeof(double) * n, hipMemcpyHostToDevice, s));
  RealAMG *G = nullptr;
  GP_TRY(real_amg_create(n, nnz, dr, dc, dv, smoother, &G, s));
  struct GGuard { RealAMG *g; ~GGuard() { real_amg_destroy(g); } } gg{G};
  scratch_trim();  // the setup's temporaries, before the 61 Krylov vectors
  int32_t it = 0;
  double rel = 0.;
  gp_status st = real_amg_solve(G, 1, bd, xd, tol, 1000, &it, &rel, s);
  if (iters_out) *iters_out = it;
  if (relres_out) *relres_out = rel;
  if (st != GP_OK && st != GP_ERR_NOCONV) return st;
  GP_HIP(hipMemcpyAsync(x, xd, sizeof(double) * n, hipMemcpyDeviceToHost, s));
  GP_HIP(hipStreamSynchronize(s));
  return st;
}

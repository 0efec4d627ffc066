// real.hpp -- device-resident real AMG + FGMRES solve, the engine under
// gp_solve_real (the hypreSolve replacement, src/hypreSolve.cpp:9-283) and
// under the V0 quasi-static path, which reuses one setup for all the solves
// with Ad or Ac (src/matrixCon.cpp:392, 511, 544).
#pragma once
#include "sparse.hpp"

namespace gp {

struct RealAMG;

// Builds the hierarchy of the n x n matrix given as device COO triplets
// (duplicates summed), smoothing with smoother (gp_real_smoother).  The
// solver owns its copy of the matrix.
gp_status real_amg_create(int64_t n, int64_t nnz, const int64_t *rows, const int64_t *cols, const double *vals,
                          int smoother, RealAMG **out, hipStream_t s);
// x = A^-1 b for k = 1, 2, 4 or 8 columns (device vectors, row i column j at
// i*k + j) by FGMRES(30) preconditioned with one V-cycle, from x = 0, until
// ||b - A x|| <= tol ||b|| or maxit iterations in every column; iters and relres
// have k entries.  Returns GP_ERR_NOCONV when a column misses the tolerance (x
// holds the last iterate).  The vectors it works on stay with the solver.
gp_status real_amg_solve(RealAMG *G, int k, const double *b, double *x, double tol, int maxit, int32_t *iters,
                         double *relres, hipStream_t s);
// y = alpha M x, or y += alpha M x, for k columns as above and value array
// `which` of M, whose rows above kLongRow must be listed (csr_mark_long); part
// holds M.nchunk * k doubles.
gp_status real_mv(const Csr &M, int which, int k, double alpha, int acc, const double *x, double *y, double *part,
                  hipStream_t s);
int64_t real_amg_rows(const RealAMG *G);
int32_t real_amg_levels(const RealAMG *G);
int64_t real_amg_bytes(const RealAMG *G);
// device bytes of a solve's vectors per column, and those held now
int64_t real_amg_column_bytes(const RealAMG *G);
int64_t real_amg_work_bytes(const RealAMG *G);
// gives a solve's vectors back (none may be running)
void real_amg_trim(RealAMG *G);
void real_amg_destroy(RealAMG *G);

}  // namespace gp

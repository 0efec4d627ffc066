// dense.hpp -- dense FP64 inverses for the coarsest levels.
#pragma once
#include <cstdint>

#include "gp_dev.hpp"

namespace gp {

template <class T>
struct C2 { T x, y; };

// a: nb row-major n x n complex matrices, overwritten by their inverses.
gp_status dense_inverse_batched(C2<double> *a, int n, int nb, hipStream_t s);
// a: one row-major real n x n matrix, overwritten by its inverse.
gp_status dense_inverse_real(double *a, int n, hipStream_t s);

// Blocks up to this many rows are inverted by one workgroup each.
constexpr int kGJWorkgroupMax = 512;

// Gauss-Jordan with partial pivoting, one workgroup per augmented matrix
// [A | I] (row-major b x 2b, device memory): count blocks listed in `list`
// (block q of b = boff[q+1] - boff[q] rows at aug + aoff[q]); bad[0] is set on a
// zero pivot column.  Asynchronous on s.
gp_status gj_workgroup(const int32_t *list, const int32_t *boff, const int64_t *aoff, int count, C2<double> *aug,
                       int *bad, hipStream_t s);

}  // namespace gp

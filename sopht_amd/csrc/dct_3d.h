// Cosine-transform passes of the fast-diagonalisation solver (dct_3d.hip).
#pragma once

#include "common.h"

namespace sopht {

struct DctPlan;  // tables of one grid: FFT twiddles, half-sample twiddles and eigenvalues per axis

// Whether a grid's axes all have a cosine-transform length.
bool dct_supported(const int64_t n[3]);
// lam[axis]: the n[axis] eigenvalues of the axis in increasing order (mode k at k).
int dct_create(int dtype, const int64_t n[3], const double* const lam[3], DctPlan** out);
void dct_destroy(DctPlan* P);
// Reals between the planes of the workspace of dct_solve: a plane and one 128-byte line, so that the
// cells of a z column spread over the memory channels (256^3: FP32 403 against 390 us per solve, FP64
// 824 against 786; 384^3 FP64 3.62 against 3.48 ms; within 1% up to 192^3).
int64_t dct_plane(int dtype, const int64_t n[3]);
// psi = V Lambda^-1 V^T rhs on ncomp contiguous (nz, ny, nx) fields through `work` (ncomp * nz
// planes); sol may be rhs. Stage marks first .. first + 4 after the five passes.
int dct_solve(DctPlan* P, void* sol, const void* rhs, void* work, int ncomp, hipStream_t s, StageTimer* tm,
              int first);

}  // namespace sopht

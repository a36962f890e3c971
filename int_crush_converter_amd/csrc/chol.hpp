// Blocked fp32 Cholesky and triangular inverse of chol.hip, for reuse by
// other kernels' drivers (the orthonormalisation of lowrank.hip).
#pragma once

#include "gemm.hpp"
#include "split.hpp"

namespace icq {

// potrf's fp64 tiles of the diagonal blocks (packed as chol.hip describes) for
// `batch` matrices of order n: their doubles, and their place from p on.
int64_t tile_doubles(int64_t batch, int64_t n);
double* tiles_at(void* p);

// Lower Cholesky in place of `batch` matrices [n, n] (pitch ld, stride sH);
// info[b] receives the 1-based column of the first non-positive pivot (or
// stays as it was).  The strict upper triangle is left as it was, except in
// the 128 x 128 diagonal blocks (zeroed).
// Lp: planes for L (SP_LOWER): the larger trailing updates are split products,
// and with `merges` the planes then hold the blocks that trtri's split merges
// read.
int potrf(float* H, int64_t batch, int64_t n, int64_t ld, int64_t sH, double* tiles, int* info, hipStream_t st,
          const SplitPlanes* Lp = nullptr, bool merges = false);

// Split planes of a large inverse: L (from potrf), X^T (whole on return), X
// by rows and the merges' intermediate products.
struct SplitWork {
    SplitPlanes L, XT, XR, T;
};

// X = L^-1 from potrf's L and tiles (the diagonal blocks inverted in fp64 and
// rounded to fp32): the lower triangle of X is exact, its strict upper
// triangle outside the diagonal blocks is scratch.
int trtri(const float* L, float* X, int64_t batch, int64_t n, int64_t ld, int64_t sH, const double* tiles,
          hipStream_t st, const SplitWork* w = nullptr);

}  // namespace icq

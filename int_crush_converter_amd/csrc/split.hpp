// fp32 products on the bf16 matrix cores: every fp32 operand x is the exact
// sum of three bf16 values x0 + x1 + x2 (8 significant bits each, rounded to
// nearest, so 24 bits in all; exact from 2^-109 on, where x2's last bit is
// still a normal bf16's, up to bf16's largest), and a product takes the six
// terms x_i y_j with i + j <= 2.  The dropped ones are at most 2^-23 |x y|
// (x1 <= 2^-8 |x|, x2 <= 2^-16 |x|); of 2e7 random pairs 2^-24 at most and
// 2^-27.5 in the root mean square, a fifth of an fp32 rounding's.  Used by the
// Hessian inverse's large products (chol.hip) and the greedy search's cross
// terms (ldlq.hip).
//
// Operands are split once, into planes laid out as the products read them:
// a chunk holds 128 rows x 16 k as [plane 3][octet 2][row 128][8 k] bf16
// (12 KB), so that a stage of a tile is one contiguous copy to LDS and an
// MFMA operand is one 16-byte LDS read.  Chunks of a row block follow each
// other along k; rows and k past the matrix hold zeros, so the products need
// no bounds checks.
#pragma once

#include "gemm.hpp"

namespace icq {

constexpr int SP_ROWS = 128;                      // rows of a chunk
constexpr int SP_K = 16;                          // k of a chunk
constexpr int64_t SP_CHUNK = 3 * SP_ROWS * SP_K;  // bf16 values of a chunk
constexpr int64_t SP_PER_BLOCK = SP_ROWS / SP_K;  // chunks along 128 k

// Which chunks (row block r, k chunk c) a set of planes holds, for a square
// matrix of nb blocks of 128: the lower triangle by rows (c < 8 (r + 1)),
// its transpose (c >= 8 r), or a rectangle of kc chunks a row block.
enum SplitKind : int { SP_LOWER = 0, SP_UPPER = 1, SP_RECT = 2 };

struct SplitPlanes {
    uint16_t* p = nullptr;
    int kind = SP_RECT;
    int64_t nb = 0;      // SP_UPPER: row blocks; SP_RECT: chunks per row block
    int64_t stride = 0;  // bf16 values between the matrices of a batch
};

__host__ __device__ inline int64_t split_chunk(const SplitPlanes& s, int64_t r, int64_t c) {
    if (s.kind == SP_LOWER) return SP_PER_BLOCK * (r * (r + 1) / 2) + c;
    if (s.kind == SP_UPPER) return SP_PER_BLOCK * (r * s.nb - r * (r - 1) / 2 - r) + c;
    return r * s.nb + c;
}

// One operand (or plane output) of a product: planes and the block (row
// block, k chunk) where it starts; launch entry z starts zr / zc further on
// and zp values of bf16 behind (pairs of one matrix, or matrices).
struct SplitOp {
    SplitPlanes s;
    int64_t r0 = 0, c0 = 0;
    int64_t zr = 0, zc = 0, zp = 0;
};

// C = alpha * A B^T over k chunks [0, kchunks) of A and B (each row-major in
// k), in 128 x 128 tiles; see split_gemm in split.hip.
struct SplitGemm {
    int64_t M, N, K;             // K: a multiple of 128 (padded with zeros)
    float alpha;                 // +1 or -1; with `sub` the result is C - A B^T
    int sub;                     // 1: C <- C - P_0 - P_1 ..., chunk of 128 k by chunk
    SplitOp A, B;
    float* C; int64_t ldc; int64_t sC;   // fp32 output (null: none)
    SplitOp out;                 // planes of C^T: rows = columns of C, k = rows of C (out.s.p null: none)
    int cmask, krange;           // CMASK_* / KR_* of gemm.hpp
    int64_t batch;
    int tag; double algo_flops;
};
int split_gemm(const SplitGemm& g, hipStream_t st);

// Planes of rows [r0, r1) x columns [c0, c1) of the fp32 matrix A (n x n, or
// n x ncols; pitch ld), by rows (transpose = 0: chunk row = row of A, k = column) or
// transposed (chunk row = column, k = row).  r0, c0 are multiples of 128;
// lower != 0: only 128-blocks on and below the diagonal.  Chunks are those
// of the whole matrix.  Elements past n (ncols) are zeros.  squares > 1: that many
// such regions, `step` rows and columns apart.
int split_planes(const float* A, int64_t n, int64_t ld, int64_t sA, int64_t r0, int64_t r1, int64_t c0, int64_t c1,
                 int transpose, int lower, const SplitPlanes& out, int64_t batch, hipStream_t st, int64_t squares = 1,
                 int64_t step = 0, int64_t ncols = -1);

}  // namespace icq

// Damped-Hessian inverse H^-1 = L^-T L^-1 (the reference's
// torch.linalg.cholesky + torch.cholesky_inverse, converter/rounding.py:19-34,
// after the damping of converter/gptq.py:91-121), for one matrix or a batch
// of equal-size diagonal blocks.
//
//  1. damp:   H += fp32(damping) * max(mean(diag H), 1e-6) * I   (per matrix)
//  2. potrf:  blocked right-looking Cholesky, nb = 128.  The nb x nb diagonal
//             block is factored by one work-group, the panel is solved with
//             it (both fp64), and the trailing update A22 -= A21 A21^T is a
//             GEMM.
//  3. trtri:  X = L^-1: the diagonal blocks' inverses (fp64), then adjacent
//             diagonal inverses merged level by level, X21 = -X22 (L21 X11)
//             (GEMMs)
//  4. lauum:  H^-1 (upper triangle) = X^T X, one GEMM whose tile (I, J)
//             only runs k >= max(I, J) because X is lower triangular.
// Flops: n^3/3 each for 2-4; all but the nb x nb factorisations are MFMA.
#include <utility>
#include <vector>

#include "chol.hpp"
#include "gemm_dev.hpp"
#include "split.hpp"
#include "torchsum.hpp"

namespace icq {

constexpr int NB = 128;

static double dtri(double n) { return n * (n + 1) / 2; }

// One work-group of 256 per matrix: H += damping * max(mean(diag H), 1e-6) * I
// with the mean computed as the reference computes H.diagonal().mean() on
// the CPU (converter/gptq.py:104, 118; ldlq.py:83, 169, 207): torch's fp32
// scalar row_sum of the strided diagonal, then one IEEE division by n.  (At
// n >= 32768 torch splits a full reduction over its CPU threads, so this is
// its one-thread order there.)  The diagonal is staged in LDS first, so
// every load is in flight at once.
constexpr int DAMP_LDS = 16384;
__global__ __launch_bounds__(256) void damp_kernel(float* H, int64_t n, int64_t ld, int64_t stride, float damping) {
    float* A = H + (int64_t)blockIdx.x * stride;
    __shared__ float dg[DAMP_LDS];
    __shared__ float blk[RS_MAX_BLOCKS];
    __shared__ float part[4];
    const bool staged = n <= DAMP_LDS;
    if (staged) {
        for (int64_t i0 = threadIdx.x; i0 < n; i0 += 8 * (int64_t)blockDim.x) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t i = i0 + u * (int64_t)blockDim.x;
                v[u] = i < n ? A[i * ld + i] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t i = i0 + u * (int64_t)blockDim.x;
                if (i < n) dg[i] = v[u];
            }
        }
    }
    __syncthreads();
    const float sum = row_sum_wg([&](int64_t i) { return staged ? dg[i] : A[i * ld + i]; }, n, blk, part);
    float mean = sum / (float)n;
    mean = mean > 1e-6f ? mean : (mean != mean ? mean : 1e-6f);
    const float delta = damping * mean;
    if (staged) {
        // the diagonal is in LDS: stores only, none waits for a load
        for (int64_t i = threadIdx.x; i < n; i += blockDim.x) A[i * ld + i] = dg[i] + delta;
        return;
    }
    for (int64_t i0 = threadIdx.x; i0 < n; i0 += 8 * (int64_t)blockDim.x) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int64_t i = i0 + u * (int64_t)blockDim.x;
            v[u] = i < n ? A[i * ld + i] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int64_t i = i0 + u * (int64_t)blockDim.x;
            if (i < n) A[i * ld + i] = v[u] + delta;
        }
    }
}

// Factor the diagonal block [k0, k0+nb) of a matrix in place (lower, upper
// part of the block set to 0) and write what the panel solve and the
// triangular inverse need of it to `tiles` (packed, below).  info[b]
// gets the 1-based column of the first non-positive pivot (LAPACK convention)
// if it is still 0.  A partial block (nb < 128) is padded with the identity.
//
// The arithmetic is fp64 (inputs and outputs fp32): the diagonal blocks feed
// every later step, and an fp64 factor and panel solve keep the whole inverse
// at the accuracy of the reference's LAPACK fp32 path.
//
// Bound by the serial chain of 128 columns on one CU.  The block is processed
// in 8 panels of 16 columns: wave 0 factors and inverts the diagonal
// tiles, six other waves (W = 1..6) own the other 16x16 tiles of the lower triangle
// (in MFMA accumulators, dealt round-robin in column-major order, so that a
// tile column has one tile per wave, the first one of a wave two).  Panel J has two phases:
//   F: wave 0 updates its copy of tile (J, J) with panel J - 1 and factors
//      it; the others apply panel J - 1's update A -= L L^T to their tiles of
//      columns >= J, hand tile (J + 1, J + 1) to wave 0 and write panel J - 1;
//   S: the owners of the tiles below it solve L_IJ^T = L_JJ^-1 A_IJ^T.
// Tiles are held transposed, so that a solved fragment (D layout) is at once
// the operand of the updates (v_mfma_f64_16x16x4_f64 throughout).  Every
// element receives its updates in panel order with the same fp64 operations,
// so the result does not depend on the schedule.
//
// MFMA 16x16x4 f64 operand layout (lane l of 64; D differs from the f32
// variant's 4*(l/16) + v):
//   A: A[i = l%16][k = l/16]      B: B[k = l/16][j = l%16]
//   D (4 doubles v): D[i = l/16 + 4*v][j = l%16]
// so a D fragment is the B operand of four MFMA steps as it stands.
//
// Packed tiles: tile (J, K), K <= J, of a block's factor at tiles +
// (J (J + 1) / 2 + K) * 256, in A-operand order with two steps adjacent:
// value [h][lane][e] is L[16 J + perm16(l%16)][16 K + 4 (l/16) + 2 h + e], and on the
// diagonal the same of L_JJ^-1.  perm16 orders the 16 indices so that the four
// that a lane's D fragment holds are adjacent in memory (4 g .. 4 g + 3).
typedef double ddoublex4 __attribute__((ext_vector_type(4)));
typedef double ddoublex2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ double rdlane(double v, int l) {
    const int64_t b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffff), l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((int64_t)hi << 32) | (uint32_t)lo);
}

// Work-group: wave 0 factors; waves 1, 2, 3, 5, 6, 7 hold tiles.  Wave 4 only
// helps to stage: it shares wave 0's SIMD, where another wave's fp64 MFMAs
// would hold its chain up (fp64 vector and matrix instructions share a unit).
constexpr int DIAG_WAVES = 8, TILE_WAVES = 6;
constexpr int DT = 16, DN = NB / DT;     // tile, tiles per side
constexpr int DIAG_TILES = DN * (DN + 1) / 2;
constexpr int DSLOTS = 6;                // tiles per MFMA wave (at most)
constexpr int64_t PACKED = DT * DT;      // doubles of a packed tile

__host__ __device__ constexpr int packed_at(int J, int K) { return J * (J + 1) / 2 + K; }
__device__ __forceinline__ constexpr int perm16(int i) { return 4 * (i & 3) + (i >> 2); }

// Lower tile `id` in column-major order over the lower triangle: tile column
// and tile row.  Tile wave W (1..6) owns the tiles id = W - 1 + 6 s.
constexpr int cm_col(int id) {
    int J = 0;
    while (id >= 8 - J) { id -= 8 - J; ++J; }
    return J;
}
constexpr int cm_row(int id) {
    int J = 0;
    while (id >= 8 - J) { id -= 8 - J; ++J; }
    return J + id;
}
constexpr int tile_id(int W, int s) { return W - 1 + TILE_WAVES * s; }

// Slot S of wave W as compile-time constants, and a loop over a wave's
// slots that hands each one to f as a type (so every tile coordinate is a
// constant and the accumulators are indexed statically).
template <int W, int S>
struct DiagSlot {
    static constexpr int s = S;
    static constexpr bool ok = tile_id(W, S) < DIAG_TILES;
    static constexpr int I = ok ? cm_row(tile_id(W, S)) : 0;
    static constexpr int J = ok ? cm_col(tile_id(W, S)) : 0;
};
template <int W, typename F, int... S>
__device__ __forceinline__ void each_slot_impl(F&& f, std::integer_sequence<int, S...>) {
    (f(DiagSlot<W, S>{}), ...);
}
template <int W, typename F>
__device__ __forceinline__ void each_slot(F&& f) {
    each_slot_impl<W>(f, std::make_integer_sequence<int, DSLOTS>{});
}

constexpr int IP = DT + 1;   // pitch of the inverse tile
constexpr int UP = NB + 4;   // pitch of the staged panel rows of the block's update

struct DiagShared {
    union {
        float P[NB * UP];         // the previous block's panel rows that update this block
        double op[DN][4][64];     // the last panel's L_IJ, operand form: [step][lane]; over the first 32 rows of
    };                            // P, which only the updates of tile columns 0 and 1 read (before the first L_IJ)
    double dg[4][64];             // the next diagonal tile, D layout
    double inv[DT][IP];           // L_JJ^-1
};
static_assert(sizeof(double) * DN * 4 * 64 <= sizeof(float) * 2 * DT * UP, "the panel's operands fit");

// The phases hand data to each other only through LDS, so they are separated
// by lds_barrier() (common.hpp), which does not wait for global stores.

// Wave 0: the Cholesky factor of the symmetric tile `acc` (D layout), as
// Lt = L^T, and X = L^-1, by rank-1 updates on the matrix cores: row c of the
// tile, scaled, is an MFMA operand where it stands (its lanes are those of one
// k), so neither the update nor the elimination of the identity needs a
// broadcast; only the pivot goes through readlane.  A column takes about 170
// cycles (420 with the panel's rows broadcast by readlane, 26 of 31 us a
// block).  col0: the tile's first column, for `bad`.
__device__ __forceinline__ void factor_tile(ddoublex4& acc, ddoublex4& Lt, ddoublex4& X, int lane, int col0,
                                            int& bad) {
    const int lr = lane >> 4, lj = lane & 15;
    ddoublex4 R;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        R[v] = lr + 4 * v == lj ? 1.0 : 0.0;
        Lt[v] = X[v] = 0.0;
    }
    double pn = 0.0, prinv = 0.0;   // the previous column's -l and 1 / sqrt(pivot)
    auto column = [&](auto cc) {
        constexpr int c = decltype(cc)::value, v = c >> 2, g = c & 3;
        const double r = acc[v];
        const double d = rdlane(r, 16 * g + c);
        double r0 = __builtin_amdgcn_rsq(d);
        __builtin_amdgcn_sched_barrier(0);
        // the previous column's elimination of the identity, behind the root
        if constexpr (c > 0) {
            constexpr int w = (c - 1) >> 2;
            const bool row = lr == ((c - 1) & 3);
            const double x = (row ? R[w] : 0.0) * prinv;
            X[w] = row ? x : X[w];
            R = __builtin_amdgcn_mfma_f64_16x16x4f64(pn, x, R, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        // l = r / sqrt(d): the hardware estimate r0 of 1/sqrt(d) (relative
        // error e/2) and one step of third order, r0 (1 + e/2 + 3/8 e^2),
        // applied to r r0; a bad pivot's root counts as 1
        const bool ok = d > 0.0;
        r0 = ok ? r0 : 1.0;
        const double rm = lr == g && lj >= c ? r : 0.0;
        double rn = -rm;
        asm volatile("" : "+v"(rn));   // l and -l side by side, not one after the other
        const double q = rm * r0, qn = rn * r0;
        double e = fma(-d * r0, r0, 1.0);
        e = ok ? e : 0.0;
        const double ep = e * fma(0.375, e, 0.5);
        const double l = fma(q, ep, q), nl = fma(qn, ep, qn);
        // (row and column c, finished, become rounding errors)
        if constexpr (c < DT - 1) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(nl, l, acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        bad = !ok && !bad ? col0 + c + 1 : bad;
        Lt[v] = lr == g ? l : Lt[v];
        pn = nl;
        prinv = fma(r0, ep, r0);
    };
    static_for<0, DT>(column);
    X[3] = lr == 3 ? R[3] * prinv : X[3];   // the last row
}

// Rows of tile (I, J) of the block from memory into D layout, transposed
// (element (row lr + 4 v of J, column lj of I) is C[16 I + lj][16 J + lr + 4 v];
// a diagonal tile is symmetric, its upper part taken from the lower), loads
// clamped into the block (no branch); outside it the identity.
__device__ __forceinline__ void load_tile(const float* A, int64_t ld, int nb, int I, int J, int lr, int lj,
                                          float (&raw)[4]) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        int i = I * DT + lj, j = J * DT + lr + 4 * v;
        if (I == J && i < j) {
            const int t = i;
            i = j;
            j = t;
        }
        const int ic = i < nb ? i : nb - 1, jc = j < nb ? j : nb - 1;
        const float x = A[(int64_t)ic * ld + jc];
        raw[v] = i < nb ? x : (i == j ? 1.0f : 0.0f);
    }
}

// The same tile of P P^T (P: the staged panel rows), fp32 products as in the
// update of the columns beside the block; added to the tile negated.  k = 16 q
// + 4 lr + s in step s: one 16-byte read per operand and four steps; the A
// operand's rows are taken in perm16 order, so that the f32 result (row
// 4 (l/16) + v) has the f64 accumulators' rows.
__device__ __forceinline__ void tile_update(const float* P, int I, int J, int lr, int lj, ddoublex4& acc) {
    gk::floatx4 u[2];
    u[0] = u[1] = gk::floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NB / 16; ++q) {
        const gk::floatx4 a = *reinterpret_cast<const gk::floatx4*>(&P[(J * DT + perm16(lj)) * UP + 16 * q + 4 * lr]);
        const gk::floatx4 b = *reinterpret_cast<const gk::floatx4*>(&P[(I * DT + lj) * UP + 16 * q + 4 * lr]);
#pragma unroll
        for (int s = 0; s < 4; ++s) u[s & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], u[s & 1], 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] -= (double)u[0][v] + (double)u[1][v];
}

// Tile wave W: the tiles below the diagonal, and the diagonal ones until they
// go to wave 0 (tile (0, 0) is there from the start).  UPD: P P^T is
// subtracted first, tile column J + 1 in phase F of panel J.
template <int W, bool UPD>
__device__ __forceinline__ void diag_tile_wave(DiagShared& sh, float* A, int64_t ld, int nb, double* packed,
                                               int lane) {
    const int lr = lane >> 4, lj = lane & 15;
    ddoublex4 acc[DSLOTS];
    float raw[DSLOTS][4];
    each_slot<W>([&](auto t) {
        using T = decltype(t);
        if constexpr (T::ok && T::I + T::J > 0) load_tile(A, ld, nb, T::I, T::J, lr, lj, raw[T::s]);
    });
    if (UPD) __syncthreads();   // sh.P
    each_slot<W>([&](auto t) {
        using T = decltype(t);
        if constexpr (T::ok && T::I + T::J > 0) {
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[T::s][v] = (double)raw[T::s][v];
            if constexpr (UPD && T::J == 0) tile_update(sh.P, T::I, T::J, lr, lj, acc[T::s]);
        }
    });
    for (int J = 0; J < DN; ++J) {
        // ---- phase F
        const double (*op)[4][64] = sh.op;   // panel J - 1
        auto apply = [&](auto t) {
            using T = decltype(t);
            double a[4], b[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                a[s] = op[T::J][s][lane];
                b[s] = op[T::I][s][lane];
            }
#pragma unroll
            for (int s = 0; s < 4; ++s)
                acc[T::s] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[s], b[s], acc[T::s], 0, 0, 0);
        };
        // the column that is solved next comes first
        each_slot<W>([&](auto t) {
            using T = decltype(t);
            if constexpr (T::ok && T::J >= 1 && T::I > T::J) {
                if (T::J == J) apply(t);
            }
        });
        if (UPD) {
            each_slot<W>([&](auto t) {
                using T = decltype(t);
                if constexpr (T::ok && T::J >= 1) {
                    if (T::J == J + 1) tile_update(sh.P, T::I, T::J, lr, lj, acc[T::s]);
                }
            });
        }
        each_slot<W>([&](auto t) {
            using T = decltype(t);
            if constexpr (T::ok && T::J >= 2) {
                if (J >= 1 && T::J > J) apply(t);
            }
            if constexpr (T::ok && T::J >= 1 && T::I == T::J) {
                if (T::J == J + 1) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) sh.dg[v][lane] = acc[T::s][v];
                }
            }
        });
        // panel J - 1 (solved, in the accumulators) to memory, its mirror zeroed
        each_slot<W>([&](auto t) {
            using T = decltype(t);
            if constexpr (T::ok && T::I > T::J) {
                if (T::J == J - 1) {
                    double* o = packed + packed_at(T::I, T::J) * PACKED;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int i = T::I * DT + lj, j = T::J * DT + lr + 4 * v;
                        if (i < nb && j < nb) A[(int64_t)i * ld + j] = (float)acc[T::s][v];
                        const int mi = T::J * DT + lr + 4 * v, mj = T::I * DT + lj;
                        if (mi < nb && mj < nb) A[(int64_t)mi * ld + mj] = 0.0f;
                        // column lr + 4 v: 4 (l/16) + 2 h + e with l/16 = v; row lj = perm16(l%16)
                        o[((lr >> 1) * 64 + 16 * v + perm16(lj)) * 2 + (lr & 1)] = acc[T::s][v];
                    }
                }
            }
        });
        lds_barrier();
        // ---- phase S
        each_slot<W>([&](auto t) {
            using T = decltype(t);
            if constexpr (T::ok && T::I > T::J) {
                if (T::J == J) {
                    double a[4];
#pragma unroll
                    for (int s = 0; s < 4; ++s) a[s] = sh.inv[lj][lr + 4 * s];
                    ddoublex4 x = ddoublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int s = 0; s < 4; ++s) x = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], acc[T::s][s], x, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) sh.op[T::I][v][lane] = x[v];
                    acc[T::s] = x;
                }
            }
        });
        lds_barrier();
    }
}

// Wave 0: the diagonal tiles.
template <bool UPD>
__device__ __forceinline__ void diag_factor_wave(DiagShared& sh, float* A, int64_t ld, int nb, double* packed,
                                                 int lane, int& bad) {
    const int lr = lane >> 4, lj = lane & 15;
    ddoublex4 acc, Lt, X;
    float raw[4];
    load_tile(A, ld, nb, 0, 0, lr, lj, raw);
    if (UPD) __syncthreads();   // sh.P
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = (double)raw[v];
    if (UPD) tile_update(sh.P, 0, 0, lr, lj, acc);
    for (int J = 0; J < DN; ++J) {
        if (J > 0) {
            const double (*op)[64] = sh.op[J];
            double a[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) a[s] = op[s][lane];
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[s], a[s], acc, 0, 0, 0);
        }
        factor_tile(acc, Lt, X, lane, J * DT, bad);
#pragma unroll
        for (int v = 0; v < 4; ++v) sh.inv[lr + 4 * v][lj] = X[v];
        lds_barrier();
        if (J + 1 < DN) {
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[v] = sh.dg[v][lane];
        }
        ddoublex2* o = reinterpret_cast<ddoublex2*>(packed + packed_at(J, J) * PACKED) + lane;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const double* q = &sh.inv[perm16(lj)][4 * lr + 2 * h];
            o[h * 64] = ddoublex2{q[0], q[1]};
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = J * DT + lj, j = J * DT + lr + 4 * v;
            if (i < nb && j < nb) A[(int64_t)i * ld + j] = (float)Lt[v];
        }
        lds_barrier();
    }
}

// The diagonal block of matrix b, by a work-group of DIAG_WAVES waves; UPD:
// updated first with the 128 columns of the panel before it (VEC: its rows
// are 16-byte aligned).
template <bool UPD, bool VEC = false>
__device__ __forceinline__ void diag_block(DiagShared& sh, int b, float* H, int64_t ld, int64_t stride, int64_t k0,
                                           int nb, double* tiles, int64_t dstride, int* info) {
    float* A = H + (int64_t)b * stride + k0 * ld + k0;
    double* packed = tiles + (int64_t)b * dstride;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // uniform
    int bad = 0;
    if (UPD) {
        // rows of the panel before the block (columns k0 - NB ..), rows past it as zeros
        const float* Pg = A - NB;
        const int r = threadIdx.x >> 5, c = (threadIdx.x & 31) * 4;
        float v[NB / 16][4];
#pragma unroll
        for (int u = 0; u < NB / 16; ++u) {
            const bool in = r + 16 * u < nb;
            const float* q = Pg + (int64_t)(in ? r + 16 * u : 0) * ld + c;
            if (VEC) {
                const float4 f = *reinterpret_cast<const float4*>(q);
                v[u][0] = f.x; v[u][1] = f.y; v[u][2] = f.z; v[u][3] = f.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[u][e] = q[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[u][e] = in ? v[u][e] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < NB / 16; ++u)
            *reinterpret_cast<float4*>(&sh.P[(r + 16 * u) * UP + c]) = make_float4(v[u][0], v[u][1], v[u][2], v[u][3]);
    }
    switch (wave) {
        case 0: diag_factor_wave<UPD>(sh, A, ld, nb, packed, lane, bad); break;
        case 1: diag_tile_wave<1, UPD>(sh, A, ld, nb, packed, lane); break;
        case 2: diag_tile_wave<2, UPD>(sh, A, ld, nb, packed, lane); break;
        case 3: diag_tile_wave<3, UPD>(sh, A, ld, nb, packed, lane); break;
        case 5: diag_tile_wave<4, UPD>(sh, A, ld, nb, packed, lane); break;
        case 6: diag_tile_wave<5, UPD>(sh, A, ld, nb, packed, lane); break;
        case 7: diag_tile_wave<6, UPD>(sh, A, ld, nb, packed, lane); break;
        default:
            if (UPD) __syncthreads();   // then gone: a barrier waits only for the waves still running
            return;
    }
    if (threadIdx.x == 0 && bad && info[b] == 0) info[b] = (int)k0 + bad;
}

__global__ __launch_bounds__(DIAG_WAVES * 64) void potrf_diag_kernel(float* H, int64_t ld, int64_t stride, int64_t k0,
                                                                    int nb, double* tiles, int64_t dstride,
                                                                    int* info) {
    __shared__ __attribute__((aligned(16))) DiagShared sh;
    diag_block<false>(sh, blockIdx.x, H, ld, stride, k0, nb, tiles, dstride, info);
}

// The diagonal block of matrix blockIdx.z (work-group 0), which it updates
// with the previous block's panel first, beside that panel's update of the
// rest of the super-block: work-group t >= 1 runs tile t (REST_T x REST_T) of
// the GEMM g (batch entry blockIdx.z; tile 0 is the diagonal block) on its
// first four waves, in the LDS the diagonal block uses; the other waves end
// at once (a barrier waits only for the waves still running).  One launch
// instead of two, and the update runs while the diagonal block's serial chain
// does.
constexpr int REST_T = 128;
static_assert(2 * gk::Geo<REST_T>::TILE_F * sizeof(float) <= sizeof(DiagShared), "GEMM tile staging fits");
template <bool VEC>
__global__ __launch_bounds__(DIAG_WAVES * 64) void potrf_diag_rest_kernel(float* H, int64_t ld, int64_t stride,
                                                                         int64_t k0, int nb, double* tiles,
                                                                         int64_t dstride, int* info, GemmArgs g) {
    __shared__ __attribute__((aligned(16))) DiagShared sh;
    if (blockIdx.x == 0) {
        diag_block<true, VEC>(sh, blockIdx.z, H, ld, stride, k0, nb, tiles, dstride, info);
        return;
    }
    if (threadIdx.x >= 256) return;
    const gk::TileRange tr = gk::tile_of<REST_T>(g, blockIdx.x);
    if (tr.skip) return;
    // whole tiles of aligned rows need no checked loads
    float* lds = reinterpret_cast<float*>(&sh);
    if (VEC && tr.i0 + REST_T <= g.M && tr.j0 + REST_T <= g.N)
        gk::gemm_tile<0, 1, false, REST_T, gk::CHUNK_SUM>(g, tr, blockIdx.z, lds);
    else
        gk::gemm_tile<0, 1, true, REST_T, gk::CHUNK_SUM>(g, tr, blockIdx.z, lds);
}

// Panel solve A21 <- A21 L^-T for the m rows below a diagonal block, in
// place, in fp64 (fp32 in and out), by tile columns: with Y = A21^T,
//   X_J = L_JJ^-1 (Y_J - sum_{K<J} L_JK X_K),
// 16 rows of A21 at a time as the 16 columns of the MFMA tiles.
// Bound by the chain of tile columns.  Work-group: `groups` such sets of rows
// in turn; wave w owns tile columns w and w + 4 of Y and, in registers, the
// packed tiles that update them.  Step K: its owner forms X_K (a D fragment
// is a B operand as it stands) and hands it over through LDS; every wave
// updates its later columns.
template <int W, bool VEC>
__device__ __forceinline__ void panel_wave(float* P, int64_t m, int64_t ld, const double* packed, int groups,
                                           double (&xs)[2][4][64], int lane) {
    const int lr = lane >> 4, lj = lane & 15;
    // L tiles of column w (K = 0 .. W) and w + 4 (K = 0 .. W + 4)
    double l0[W + 1][4], l1[W + 5][4];
    auto load = [&](double (&o)[4], int J, int K) {
        const ddoublex2* q = reinterpret_cast<const ddoublex2*>(packed + packed_at(J, K) * PACKED) + lane;
        const ddoublex2 a = q[0], c = q[64];
        o[0] = a[0];
        o[1] = a[1];
        o[2] = c[0];
        o[3] = c[1];
    };
#pragma unroll
    for (int K = 0; K <= W; ++K) load(l0[K], W, K);
#pragma unroll
    for (int K = 0; K <= W + 4; ++K) load(l1[K], W + 4, K);
    for (int g = 0; g < groups; ++g) {
        const int64_t row = ((int64_t)blockIdx.x * groups + g) * 16 + lj;
        const bool in = row < m;
        float* R = P + (in ? row : 0) * ld + 4 * lr;   // this lane's columns of a tile column: 4 lr .. 4 lr + 3
        ddoublex4 y[2];
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            float v[4];
            if (VEC) {
                const float4 f = *reinterpret_cast<const float4*>(R + (W + 4 * o) * DT);
                v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = R[(W + 4 * o) * DT + e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) y[o][e] = in ? (double)v[e] : 0.0;
        }
        // X = L_KK^-1 y, to LDS and (fp32) to memory
        auto solve = [&](int K, const double (&inv)[4], const ddoublex4& yk, ddoublex4& x) {
            x = ddoublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int s = 0; s < 4; ++s) x = __builtin_amdgcn_mfma_f64_16x16x4f64(inv[s], yk[s], x, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) xs[K & 1][v][lane] = x[v];
        };
        auto store = [&](int K, const ddoublex4& x) {
            if (!in) return;
            if (VEC) {
                *reinterpret_cast<float4*>(R + K * DT) =
                    make_float4((float)x[0], (float)x[1], (float)x[2], (float)x[3]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) R[K * DT + e] = (float)x[e];
            }
        };
        auto update = [&](const double (&l)[4], const double (&x)[4], ddoublex4& yj) {
#pragma unroll
            for (int s = 0; s < 4; ++s) yj = __builtin_amdgcn_mfma_f64_16x16x4f64(-l[s], x[s], yj, 0, 0, 0);
        };
        auto step = [&](auto kc) {
            constexpr int K = decltype(kc)::value;
            ddoublex4 x;
            if constexpr (K == W) solve(K, l0[W], y[0], x);
            if constexpr (K == W + 4) solve(K, l1[W + 4], y[1], x);
            lds_barrier();
            if constexpr (K == W || K == W + 4) store(K, x);
            if constexpr (K < W + 4) {
                double xk[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) xk[v] = xs[K & 1][v][lane];
                if constexpr (K < W) update(l0[K < W ? K : 0], xk, y[0]);
                update(l1[K], xk, y[1]);
            }
        };
        static_for<0, DN>(step);
    }
}

template <bool VEC>
__global__ __launch_bounds__(256) void panel_solve_kernel(float* A21, int64_t m, int64_t ld, int64_t stride,
                                                         const double* tiles, int64_t dstride, int groups) {
    __shared__ double xs[2][4][64];
    float* P = A21 + (int64_t)blockIdx.y * stride;
    const double* packed = tiles + (int64_t)blockIdx.y * dstride;
    const int lane = threadIdx.x & 63;
    switch (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {
        case 0: panel_wave<0, VEC>(P, m, ld, packed, groups, xs, lane); break;
        case 1: panel_wave<1, VEC>(P, m, ld, packed, groups, xs, lane); break;
        case 2: panel_wave<2, VEC>(P, m, ld, packed, groups, xs, lane); break;
        default: panel_wave<3, VEC>(P, m, ld, packed, groups, xs, lane); break;
    }
}

// Diagonal blocks of X = L^-1 (128 x 128, fp32, upper part 0) from the packed
// tiles: block column J on wave J,
//   X_JJ = L_JJ^-1,  X_IJ = -L_II^-1 sum_{K=J}^{I-1} L_IK X_KJ,
// each X fragment being the B operand of the products below it.
template <int J>
__device__ __forceinline__ void dinv_wave(float* P, int64_t ld, int nb, const double* packed, int lane) {
    const int lr = lane >> 4, lj = lane & 15;
    auto store = [&](int I, const ddoublex4& x) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = I * DT + 4 * lr + v, j = J * DT + lj;
            if (i < nb && j < nb) P[(int64_t)i * ld + j] = (float)x[v];
        }
    };
    auto load = [&](int I, int K, double (&o)[4]) {
        const ddoublex2* q = reinterpret_cast<const ddoublex2*>(packed + packed_at(I, K) * PACKED) + lane;
        const ddoublex2 a = q[0], c = q[64];
        o[0] = a[0];
        o[1] = a[1];
        o[2] = c[0];
        o[3] = c[1];
    };
    for (int I = 0; I < J; ++I) store(I, ddoublex4{0.0, 0.0, 0.0, 0.0});
    ddoublex4 x[DN];
    // L_JJ^-1, row 4 lr + v (D row lr + 4 v in perm16 order), column lj
    {
        const double* q = packed + packed_at(J, J) * PACKED;
#pragma unroll
        for (int v = 0; v < 4; ++v)
            x[J][v] = q[((lj >> 1 & 1) * 64 + (lj >> 2) * 16 + (lr + 4 * v)) * 2 + (lj & 1)];
    }
    store(J, x[J]);
#pragma unroll
    for (int I = J + 1; I < DN; ++I) {
        ddoublex4 s = ddoublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int K = J; K < I; ++K) {
            double l[4];
            load(I, K, l);
#pragma unroll
            for (int u = 0; u < 4; ++u) s = __builtin_amdgcn_mfma_f64_16x16x4f64(l[u], x[K][u], s, 0, 0, 0);
        }
        double l[4];
        load(I, I, l);
        x[I] = ddoublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int u = 0; u < 4; ++u) x[I] = __builtin_amdgcn_mfma_f64_16x16x4f64(-l[u], s[u], x[I], 0, 0, 0);
        store(I, x[I]);
    }
}

__global__ __launch_bounds__(512) void dinv_kernel(float* X, int64_t n, int64_t ld, int64_t stride,
                                                  const double* tiles, int64_t dstride) {
    const int64_t k0 = (int64_t)blockIdx.x * NB;
    const double* packed = tiles + (int64_t)blockIdx.y * dstride + (int64_t)blockIdx.x * NB * NB;
    float* P = X + (int64_t)blockIdx.y * stride + k0 * ld + k0;
    const int nb = (int)std::min<int64_t>(NB, n - k0), lane = threadIdx.x & 63;
    switch (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) {
        case 0: dinv_wave<0>(P, ld, nb, packed, lane); break;
        case 1: dinv_wave<1>(P, ld, nb, packed, lane); break;
        case 2: dinv_wave<2>(P, ld, nb, packed, lane); break;
        case 3: dinv_wave<3>(P, ld, nb, packed, lane); break;
        case 4: dinv_wave<4>(P, ld, nb, packed, lane); break;
        case 5: dinv_wave<5>(P, ld, nb, packed, lane); break;
        case 6: dinv_wave<6>(P, ld, nb, packed, lane); break;
        default: dinv_wave<7>(P, ld, nb, packed, lane); break;
    }
}

// Copy the upper triangle onto the lower one (in place), per matrix, in
// 32 x 32 tiles through LDS: both the upper source tile and the lower target
// tile are read and written along rows.  Grid (tiles, tiles, batch), block
// (32, 8); work-groups above the diagonal exit.
__global__ void mirror_upper_tiled_kernel(float* H, int64_t n, int64_t ld, int64_t stride) {
    const int ti = blockIdx.y, tj = blockIdx.x;   // target tile: rows ti, columns tj (ti >= tj)
    if (ti < tj) return;
    __shared__ float S[32][33];
    float* A = H + (int64_t)blockIdx.z * stride;
    const int tx = threadIdx.x, ty = threadIdx.y;
    for (int r = ty; r < 32; r += 8) {   // source: rows tj, columns ti (upper)
        const int64_t i = (int64_t)tj * 32 + r, j = (int64_t)ti * 32 + tx;
        if (i < n && j < n) S[r][tx] = A[i * ld + j];
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int64_t i = (int64_t)ti * 32 + r, j = (int64_t)tj * 32 + tx;
        if (i < n && j < n && i > j) A[i * ld + j] = S[tx][r];
    }
}

static int mirror_upper(float* H, int64_t batch, int64_t n, int64_t ld, int64_t stride, hipStream_t st) {
    IC_REQUIRE(batch <= 65535 && cdiv(n, 32) < 65536, "mirror_upper: too large");
    const dim3 tg((unsigned)cdiv(n, 32), (unsigned)cdiv(n, 32), (unsigned)batch);
    hipLaunchKernelGGL(mirror_upper_tiled_kernel, tg, dim3(32, 8), 0, st, H, n, ld, stride);
    IC_CHECK_LAUNCH();
    return IC_OK;
}

// Transpose the lower triangle into the upper one and zero the lower (in place):
// turns a lower Cholesky factor L into L^T.
__global__ void lower_to_upper_kernel(float* H, int64_t n, int64_t ld, int64_t stride) {
    float* A = H + (int64_t)blockIdx.z * stride;
    const int64_t i = (int64_t)blockIdx.y * 16 + threadIdx.y;
    const int64_t j = (int64_t)blockIdx.x * 16 + threadIdx.x;
    if (i < n && j < n && i < j) {
        A[i * ld + j] = A[j * ld + i];
        A[j * ld + i] = 0.0f;
    }
}

int64_t tile_doubles(int64_t batch, int64_t n) { return batch * cdiv(n, NB) * NB * NB; }

double* tiles_at(void* p) {
    return reinterpret_cast<double*>((reinterpret_cast<uintptr_t>(p) + 255) & ~(uintptr_t)255);
}

// Lower Cholesky in place of `batch` matrices [n, n] (pitch ld, stride sH);
// tiles receives every block's packed tiles (batch x nblk x NB x NB doubles).
//
// Two-level right-looking: columns are taken in super-blocks of up to
// SUPER_NB columns.  After each block's panel, only the rest of the
// super-block's columns are updated (rank-NB); after the super-block, the
// trailing matrix beyond it gets one SYRK with K = SUPER_NB.  Same flops as
// one SYRK per block, with the trailing matrix read and written once per
// super-block.
//
// Inside a super-block a block costs two launches: its diagonal block, beside
// the previous block's update of the rest of the super-block (which the
// diagonal block's work-group applies to the block itself first), and its
// panel.
constexpr int64_t SUPER_NB = 1024;
constexpr int64_t PANEL_GROUPS = 512;   // two work-groups per CU

// Where the split products (split.hpp) are taken instead of gemm_f32's, by
// the matrix's order alone (a batch's matrices equal each one by itself):
// - merges of segments of SPLIT_SEG and more, in matrices of more than one.
//   The level of 1024 measured 64 us in fp32 and 99 us split at 4096 (too few
//   128-tiles), 136 and 201 us at 12288; that of 2048 187 and 173 us at 4096,
//   484 and 347 us at 12288.  X^T X: 63 and 85 us at 2048, 198 and 118 us at
//   2901 (rows that are not aligned), 242 and 194 us at 4096.
// - trailing updates of at least SPLIT_SYRK_BLOCKS blocks of rows (K = 1024,
//   splitting included): 45 and 59 us at 853 rows, 60 and 62 us at 2048 (76
//   and 63 us at 1976 rows, not aligned), 170 and 134 us at 4096.
constexpr int64_t SPLIT_SEG = 2048;
constexpr int64_t SPLIT_SYRK_BLOCKS = 15;

int potrf(float* H, int64_t batch, int64_t n, int64_t ld, int64_t sH, double* tiles, int* info, hipStream_t st,
          const SplitPlanes* Lp, bool merges) {
    const int64_t nblk = cdiv(n, NB);
    const int64_t dstride = nblk * NB * NB;
    IC_REQUIRE(batch <= 65535, "potrf: batch too large");
    const bool aligned = (uintptr_t)H % 16 == 0 && ld % 4 == 0 && sH % 4 == 0;
    bool rest_pending = false;   // `rest`: the previous block's update of its super-block, diagonal block included
    GemmArgs rest{};
    int64_t rest_tiles = 0;
    for (int64_t s0 = 0; s0 < n; s0 += SUPER_NB) {
        const int64_t s1 = std::min<int64_t>(n, s0 + SUPER_NB);
        for (int64_t k0 = s0; k0 < s1; k0 += NB) {
            const int64_t kb = k0 / NB;
            const int nb = (int)std::min<int64_t>(NB, n - k0);
            double* packed = tiles + kb * NB * NB;
            {
                double fl = batch * (2.0 / 3.0) * nb * nb * nb, by = batch * 3.0 * 4 * nb * nb;
                if (rest_pending) fl += rest.algo_flops, by += 4.0 * batch * (2.0 * rest.M * rest.K + 2.0 * rest.M * rest.N);
                ProfScope prof_scope(st, PT_DIAG, fl, by);
                const dim3 gd((unsigned)rest_tiles, 1, (unsigned)batch), wg(DIAG_WAVES * 64);
                if (rest_pending && aligned)
                    hipLaunchKernelGGL((potrf_diag_rest_kernel<true>), gd, wg, 0, st, H, ld, sH, k0, nb, packed, dstride,
                                       info, rest);
                else if (rest_pending)
                    hipLaunchKernelGGL((potrf_diag_rest_kernel<false>), gd, wg, 0, st, H, ld, sH, k0, nb, packed, dstride,
                                       info, rest);
                else
                    hipLaunchKernelGGL(potrf_diag_kernel, dim3((unsigned)batch), wg, 0, st, H, ld, sH, k0, nb, packed,
                                       dstride, info);
                IC_CHECK_LAUNCH();
                rest_pending = false;
            }
            const int64_t k1 = k0 + nb;
            const int64_t m = n - k1;
            if (m <= 0) break;
            float* A21 = H + k1 * ld + k0;
            {
                // panel: A21 <- A21 L_kk^-T (in place); at most PANEL_GROUPS work-groups, which then take
                // several sets of rows each
                ProfScope prof_scope(st, PT_PANEL, (double)batch * m * nb * (nb + 1), (double)batch * m * nb * 8.0);
                const int64_t sets = cdiv(m, 16);
                const int groups = (int)cdiv(sets, PANEL_GROUPS);
                const dim3 gd((unsigned)cdiv(sets, groups), (unsigned)batch);
                if (aligned)
                    hipLaunchKernelGGL((panel_solve_kernel<true>), gd, dim3(256), 0, st, A21, m, ld, sH, packed, dstride,
                                       groups);
                else
                    hipLaunchKernelGGL((panel_solve_kernel<false>), gd, dim3(256), 0, st, A21, m, ld, sH, packed, dstride,
                                       groups);
                IC_CHECK_LAUNCH();
            }
            // rest of the super-block: A[k1:, k1:s1] -= A21 A21[:s1-k1]^T (lower in its top square), in the next
            // diagonal block's launch.  One chunk (K = nb <= kc): C - P in the sum form, as gemm_f32 runs it
            const int64_t w = s1 - k1;
            if (w > 0) {
                rest = GemmArgs{m, w, nb, -1.0f, 1.0f, A21, ld, sH, A21, ld, sH, H + k1 * ld + k1, ld, sH, 0, 1,
                                CMASK_LOWER, KR_FULL, batch, PT_GEMM_CHOL,
                                (double)batch * 2.0 * (dtri((double)w) + (double)(m - w) * w) * nb};
                bool tri;
                rest_tiles = gk::tile_count<REST_T>(rest, tri);
                IC_REQUIRE(rest_tiles < (1LL << 30), "potrf: problem too large");
                rest_pending = true;
            }
        }
        // beyond the super-block: A[s1:, s1:] -= L[s1:, s0:s1] L[s1:, s0:s1]^T (lower)
        const int64_t m = n - s1;
        if (m > 0) {
            const float* P = H + s1 * ld + s0;
            const int64_t k = s1 - s0;
            const bool split = Lp && cdiv(m, SP_ROWS) >= SPLIT_SYRK_BLOCKS;
            if (split || (Lp && merges)) {
                // the rows that this update or a merge reads
                const int64_t r = split ? s1 : cdiv(s1, SPLIT_SEG) * SPLIT_SEG;
                int rc = split_planes(H, n, ld, sH, r, n, s0, s1, 0, 0, *Lp, batch, st);
                if (rc) return rc;
            }
            if (split) {
                SplitOp a;
                a.s = *Lp;
                a.r0 = s1 / SP_ROWS;
                a.c0 = s0 / SP_K;
                a.zp = Lp->stride;
                SplitGemm g{m, m, k, -1.0f, 1, a, a, H + s1 * ld + s1, ld, sH, SplitOp{}, CMASK_LOWER, KR_FULL, batch,
                            PT_SPLIT_CHOL, (double)batch * 2.0 * dtri((double)m) * k};
                int rc = split_gemm(g, st);
                if (rc) return rc;
                continue;
            }
            GemmArgs g{m, m, k, -1.0f, 1.0f, P, ld, sH, P, ld, sH, H + s1 * ld + s1, ld, sH, 0, 1, CMASK_LOWER,
                       KR_FULL, batch, PT_GEMM_CHOL, (double)batch * 2.0 * dtri((double)m) * k};
            g.chunk_sub = 1;
            int rc = gemm_f32(g, st);
            if (rc) return rc;
        }
    }
    return IC_OK;
}

// X = L^-1 (lower triangle and the 128x128 diagonal blocks exact; the rest
// of the upper triangle is scratch) from L (lower, in H) and the diagonal
// blocks' packed tiles, of which dinv_kernel forms X's diagonal blocks; then
// adjacent diagonal inverses are merged level by level,
//     [L11 0; L21 L22]^-1 = [X11 0; X21 X22],   X21 = -X22 (L21 X11),
// with T (or T^T when the halves differ in size) parked in the unused
// upper block of the merged square.  All pairs of one level that have the same shape run as one
// batched GEMM, so the whole inverse takes ~2 log2(n/128) launches of
// large-K GEMMs instead of 2 n/128 rank-128 updates.
static int merge_pairs(const float* L, float* X, int64_t ld, int64_t r0, int64_t n1, int64_t n2, int64_t count,
                       int64_t pstride, int64_t batch, int64_t sH, hipStream_t st) {
    // per (pair, matrix): strides differ only when both are > 1; then loop over matrices
    const bool pairs_batched = count > 1;
    const int64_t gb = pairs_batched ? count : batch;
    const int64_t gs = pairs_batched ? pstride : sH;
    const int64_t outer = pairs_batched ? batch : 1;
    for (int64_t m = 0; m < outer; ++m) {
        const int64_t off = pairs_batched ? m * sH : 0;
        const float* X11 = X + off + r0 * ld + r0;
        const float* L21 = L + off + (r0 + n1) * ld + r0;
        const float* X22 = X + off + (r0 + n1) * ld + (r0 + n1);
        float* X21 = X + off + (r0 + n1) * ld + r0;
        int rc;
        if (n2 <= n1 && n2 % NB == 0) {
            // T = L21 X11 (n2 x n1) in the upper triangle of the merged square:
            // rows r0 .. r0+n2, columns r0+n2 .. r0+n2+n1 (strictly above the
            // diagonal blocks, since n2 is a whole number of blocks; X11 is
            // read only on and below its diagonal blocks)
            float* T = X + off + r0 * ld + (r0 + n2);
            GemmArgs t{n2, n1, n1, 1.0f, 0.0f, L21, ld, gs, X11, ld, gs, T, ld, gs, 0, 0, CMASK_FULL, KR_FROM_J, gb,
                       PT_GEMM_INV, (double)gb * n2 * n1 * (n1 + 1)};
            if ((rc = gemm_f32(t, st))) return rc;
            // X21 = -X22 T; k <= i (X22 lower)
            GemmArgs x{n2, n1, n2, -1.0f, 0.0f, X22, ld, gs, T, ld, gs, X21, ld, gs, 0, 0, CMASK_FULL, KR_TO_I, gb,
                       PT_GEMM_INV, (double)gb * n1 * n2 * (n2 + 1)};
            if ((rc = gemm_f32(x, st))) return rc;
        } else {
            // T^T[a][b] = sum_k X11[k][a] L21[b][k], k >= a (X11 lower), stored n1 x n2
            float* U = X + off + r0 * ld + (r0 + n1);
            GemmArgs t{n1, n2, n1, 1.0f, 0.0f, X11, ld, gs, L21, ld, gs, U, ld, gs, 1, 1, CMASK_FULL, KR_FROM_I, gb,
                       PT_GEMM_INV, (double)gb * n2 * n1 * (n1 + 1)};
            if ((rc = gemm_f32(t, st))) return rc;
            // X21 = -X22 T, k <= i (X22 lower)
            GemmArgs x{n2, n1, n2, -1.0f, 0.0f, X22, ld, gs, U, ld, gs, X21, ld, gs, 0, 1, CMASK_FULL, KR_TO_I, gb,
                       PT_GEMM_INV, (double)gb * n1 * n2 * (n2 + 1)};
            if ((rc = gemm_f32(x, st))) return rc;
        }
    }
    return IC_OK;
}

// The same merge from L's planes, for segments of SPLIT_SEG and more: X11's
// planes are there (transposed), X22's are formed here (by rows), T stays in
// planes, and X21 is written in fp32 (a later merge's X22) and, transposed,
// beside X11's planes.
static int merge_pairs_split(float* X, int64_t n, int64_t ld, int64_t r0, int64_t n1, int64_t n2, int64_t count,
                             int64_t batch, int64_t sH, const SplitWork& w, hipStream_t st) {
    const bool pairs_batched = count > 1;
    const int64_t gb = pairs_batched ? count : batch;
    const int64_t outer = pairs_batched ? batch : 1;
    const int64_t step = pairs_batched ? n1 + n2 : 0;          // rows between the pairs
    const int64_t b0 = r0 / SP_ROWS, b1 = (r0 + n1) / SP_ROWS, n2p = cdiv(n2, SP_ROWS) * SP_ROWS;
    SplitPlanes T = w.T;
    T.nb = n2p / SP_K;
    const int64_t tz = pairs_batched ? n1 / SP_ROWS * T.nb * SP_CHUNK : T.stride;
    int rc0 = split_planes(X, n, ld, sH, r0 + n1, r0 + n1 + n2, r0 + n1, r0 + n1 + n2, 0, 1, w.XR, batch, st,
                           count, count > 1 ? n1 + n2 : 0);
    if (rc0) return rc0;
    for (int64_t m = 0; m < outer; ++m) {
        const int64_t off = pairs_batched ? m : 0;
        auto op = [&](SplitPlanes s, int64_t rb, int64_t kb) {
            SplitOp o;
            o.s = s;
            o.s.p += off * s.stride;
            o.r0 = rb;
            o.c0 = kb * SP_PER_BLOCK;
            o.zr = step / SP_ROWS;
            o.zc = step / SP_K;
            o.zp = pairs_batched ? 0 : s.stride;
            return o;
        };
        SplitOp t = op(T, 0, 0);
        t.zr = t.zc = 0;
        t.zp = tz;
        int rc;
        // T = L21 X11 (k >= column: X11 is lower)
        SplitGemm g1{n2, n1, n1, 1.0f, 0, op(w.L, b1, b0), op(w.XT, b0, b0), nullptr, 0, 0, t, CMASK_FULL, KR_FROM_J,
                     gb, PT_SPLIT_INV, (double)gb * n2 * n1 * (n1 + 1)};
        if ((rc = split_gemm(g1, st))) return rc;
        // X21 = -X22 T (k <= row: X22 is lower)
        SplitGemm g2{n2, n1, n2p, -1.0f, 0, op(w.XR, b1, b1), t, X + off * sH + (r0 + n1) * ld + r0, ld,
                     pairs_batched ? step * (ld + 1) : sH, op(w.XT, b0, b1), CMASK_FULL, KR_TO_I, gb, PT_SPLIT_INV,
                     (double)gb * n1 * n2 * (n2 + 1)};
        if ((rc = split_gemm(g2, st))) return rc;
    }
    return IC_OK;
}

int trtri(const float* L, float* X, int64_t batch, int64_t n, int64_t ld, int64_t sH, const double* tiles,
          hipStream_t st, const SplitWork* w) {
    const int64_t nblk = cdiv(n, NB);
    const int64_t dstride = nblk * NB * NB;
    hipLaunchKernelGGL(dinv_kernel, dim3((unsigned)nblk, (unsigned)batch), dim3(512), 0, st, X, n, ld, sH, tiles,
                       dstride);
    IC_CHECK_LAUNCH();
    // segments of rows [start, start + len); merged pairwise per level
    std::vector<int64_t> seg;
    for (int64_t k = 0; k < nblk; ++k) seg.push_back(k * NB);
    seg.push_back(n);
    bool split = false;   // the segments' planes exist
    while (seg.size() > 2) {
        if (w && !split && seg[1] == SPLIT_SEG) {
            int rc = split_planes(X, n, ld, sH, 0, seg[1], 0, seg[1], 1, 1, w->XT, batch, st,
                                  (int64_t)seg.size() - 1, seg[1]);
            if (rc) return rc;
            split = true;
        }
        const int64_t nseg = (int64_t)seg.size() - 1;
        const int64_t npair = nseg / 2;
        std::vector<int64_t> next;
        // pairs with the shape of the first one and uniform spacing run together
        int64_t p = 0;
        while (p < npair) {
            const int64_t r0 = seg[2 * p], n1 = seg[2 * p + 1] - r0, n2 = seg[2 * p + 2] - seg[2 * p + 1];
            int64_t q = p + 1;
            while (q < npair && seg[2 * q + 1] - seg[2 * q] == n1 && seg[2 * q + 2] - seg[2 * q + 1] == n2 &&
                   seg[2 * q] - seg[2 * q - 2] == n1 + n2)
                ++q;
            int rc = split ? merge_pairs_split(X, n, ld, r0, n1, n2, q - p, batch, sH, *w, st)
                           : merge_pairs(L, X, ld, r0, n1, n2, q - p, (n1 + n2) * (ld + 1), batch, sH, st);
            if (rc) return rc;
            p = q;
        }
        for (int64_t i = 0; i < npair; ++i) next.push_back(seg[2 * i]);
        if (nseg % 2) next.push_back(seg[nseg - 1]);
        next.push_back(n);
        seg.swap(next);
    }
    return IC_OK;
}

}  // namespace icq

using namespace icq;

// Split planes of `batch` inverses of order n: their bytes, and (w) their
// places from `base` on.
static int64_t split_bytes(int64_t batch, int64_t n, char* base, SplitWork* w) {
    const int64_t nb = cdiv(n, SP_ROWS);
    const int64_t tri = SP_PER_BLOCK * (nb * (nb + 1) / 2) * SP_CHUNK;
    const int64_t rect = SP_PER_BLOCK * (nb * nb / 4 + nb) * SP_CHUNK;   // n1 n2 <= n^2 / 4, whole blocks
    if (w) {
        uint16_t* p = reinterpret_cast<uint16_t*>(base);
        w->L = SplitPlanes{p, SP_LOWER, nb, tri};
        w->XT = SplitPlanes{p + batch * tri, SP_UPPER, nb, tri};
        w->XR = SplitPlanes{p + 2 * batch * tri, SP_LOWER, nb, tri};
        w->T = SplitPlanes{p + 3 * batch * tri, SP_RECT, 0, rect};
    }
    return batch * (3 * tri + rect) * (int64_t)sizeof(uint16_t);
}

// The planes take 10.5 n^2 bytes a matrix (three triangles of 3 n^2, n^2 / 4 of
// products at 6 bytes) beside the 8 n^2 of H and X: matrices beyond SPLIT_MAX_N
// (45 GB of planes) are inverted without them, and a batch in pieces whose
// planes take SPLIT_MAX_BYTES at most, or what room the workspace has.
constexpr int64_t SPLIT_MAX_N = 65536, SPLIT_MAX_BYTES = 64LL << 30;
// Up to SPLIT_ALIGNED_N the fp32 kernels keep up where their rows are aligned
// (a layer with a 3072 x 3072 Hessian 4.03 ms, 4.08 split); where they are not
// they do not (2901, Cholesky method: 4.13 ms, 4.05 split).  Around both lines
// the two are as fast and the split products are more precise, so that they
// begin where they cost 1.4 % at most.  Inverses, split over fp32 products: not
// aligned 2049 1.003, 2301 1.008, 2501 0.984, 2701 0.964, 3071 0.925; aligned
// 3076 0.908, 3136 1.014, 3200 1.005, 3456 1.004, 3584 0.997, 3840 0.976, 4096
// 0.967, 5120 0.918.
constexpr int64_t SPLIT_ALIGNED_N = 3072;
static bool splits(int64_t n) {
    return n > (n % 4 == 0 ? SPLIT_ALIGNED_N : SPLIT_SEG) && n <= SPLIT_MAX_N;
}
// Matrices of a batch that are inverted at once, their planes in `room` bytes
// (0: without planes).
static int64_t split_batch(int64_t batch, int64_t n, int64_t room) {
    if (!splits(n)) return 0;
    return std::min(batch, std::min(room - 256, SPLIT_MAX_BYTES) / split_bytes(1, n, nullptr, nullptr));
}

extern "C" int64_t ic_hessian_inverse_min_workspace_bytes(int64_t batch, int64_t n) {
    return batch * n * n * (int64_t)sizeof(float) + tile_doubles(batch, n) * (int64_t)sizeof(double) + 256;
}

extern "C" int64_t ic_hessian_inverse_workspace_bytes(int64_t batch, int64_t n) {
    const int64_t step = split_batch(batch, n, INT64_MAX);
    return ic_hessian_inverse_min_workspace_bytes(batch, n) +
           (step > 0 ? split_bytes(step, n, nullptr, nullptr) + 256 : 0);
}

// `batch` damped matrices H -> their inverses (ic_hessian_inverse's methods);
// X: batch n^2 floats.
static int inverse(float* H, int64_t batch, int64_t n, int method, int* info, int* info2, float* X, double* tiles,
                   const SplitWork* w, hipStream_t st) {
    const int64_t ld = n, sH = n * n;
    const SplitPlanes* Lp = w ? &w->L : nullptr;
    int rc = potrf(H, batch, n, ld, sH, tiles, info, st, Lp, true);
    if (rc) return rc;
    rc = trtri(H, X, batch, n, ld, sH, tiles, st, w);
    if (rc) return rc;
    // H^-1 (upper triangle incl. diagonal) = X^T X  -> H
    const double flops = (double)batch * 2.0 * (double)n * (n + 1) * (n + 2) / 6.0;
    if (w) {
        SplitOp x;
        x.s = w->XT;
        x.zp = w->XT.stride;
        SplitGemm u{n, n, cdiv(n, SP_ROWS) * SP_ROWS, 1.0f, 0, x, x, H, ld, sH, SplitOp{}, CMASK_UPPER, KR_FROM_MAXIJ,
                    batch, PT_SPLIT_INV, flops};
        rc = split_gemm(u, st);
    } else {
        GemmArgs u{n, n, n, 1.0f, 0.0f, X, ld, sH, X, ld, sH, H, ld, sH, 1, 0, CMASK_UPPER, KR_FROM_MAXIJ, batch,
                   PT_GEMM_INV, flops};
        rc = gemm_f32(u, st);
    }
    if (rc) return rc;
    if (method == 2) return IC_OK;   // the lower part keeps L: finite, never read by such callers
    if ((rc = mirror_upper(H, batch, n, ld, sH, st))) return rc;
    if (method == 1) {
        // upper Cholesky factor of H^-1 (converter/gptq.py:91-110): L2 = chol(H^-1), return L2^T
        rc = potrf(H, batch, n, ld, sH, tiles, info2, st, Lp, false);
        if (rc) return rc;
        dim3 tb(16, 16), tg((unsigned)cdiv(n, 16), (unsigned)cdiv(n, 16), (unsigned)batch);
        hipLaunchKernelGGL(lower_to_upper_kernel, tg, tb, 0, st, H, n, ld, sH);
        IC_CHECK_LAUNCH();
    }
    return IC_OK;
}

extern "C" int ic_hessian_inverse_sized(float* H, int64_t batch, int64_t n, float damping, int method, int* info,
                                        void* workspace, int64_t workspace_bytes, void* stream) {
    IC_REQUIRE(H && info && workspace, "ic_hessian_inverse: null pointer");
    IC_REQUIRE(n >= 0 && batch >= 0, "ic_hessian_inverse: bad size");
    IC_REQUIRE(method >= 0 && method <= 2,
               "ic_hessian_inverse: method must be 0 (hinv), 1 (cholesky) or 2 (hinv, upper triangle)");
    if (n == 0 || batch == 0) return IC_OK;
    const int64_t least = ic_hessian_inverse_min_workspace_bytes(batch, n);
    IC_REQUIRE(workspace_bytes >= least, "ic_hessian_inverse: workspace too small");
    hipStream_t st = as_stream(stream);
    const int64_t sH = n * n;
    float* X = reinterpret_cast<float*>(workspace);
    double* tiles = tiles_at(X + batch * sH);
    IC_CHECK_HIP(hipMemsetAsync(info, 0, batch * sizeof(int), st));
    hipLaunchKernelGGL(damp_kernel, dim3((unsigned)batch), dim3(256), 0, st, H, n, n, sH, damping);
    IC_CHECK_LAUNCH();
    const int64_t step = split_batch(batch, n, workspace_bytes - least);
    if (step <= 0) return inverse(H, batch, n, method, info, info + batch, X, tiles, nullptr, st);
    const uintptr_t end = reinterpret_cast<uintptr_t>(tiles + tile_doubles(batch, n));
    char* planes = reinterpret_cast<char*>((end + 255) & ~(uintptr_t)255);
    for (int64_t b = 0; b < batch; b += step) {
        const int64_t m = std::min(step, batch - b);
        SplitWork w;
        split_bytes(m, n, planes, &w);
        int rc = inverse(H + b * sH, m, n, method, info + b, info + batch + b, X + b * sH,
                         tiles + tile_doubles(b, n), &w, st);
        if (rc) return rc;
    }
    return IC_OK;
}

extern "C" int ic_hessian_inverse(float* H, int64_t batch, int64_t n, float damping, int method, int* info,
                                  void* workspace, void* stream) {
    return ic_hessian_inverse_sized(H, batch, n, damping, method, info, workspace,
                                    ic_hessian_inverse_workspace_bytes(batch, n), stream);
}

extern "C" int ic_damp_hessian(float* H, int64_t batch, int64_t n, float damping, void* stream) {
    IC_REQUIRE(H || batch == 0 || n == 0, "ic_damp_hessian: null pointer");
    IC_REQUIRE(n >= 0 && batch >= 0 && batch < (1LL << 31), "ic_damp_hessian: bad size");
    if (n == 0 || batch == 0) return IC_OK;
    hipLaunchKernelGGL(damp_kernel, dim3((unsigned)batch), dim3(256), 0, as_stream(stream), H, n, n, n * n, damping);
    IC_CHECK_LAUNCH();
    return IC_OK;
}

extern "C" int ic_gram_tn(const float* W, int64_t M, int64_t N, int64_t ldw, float alpha, float* C, void* stream) {
    IC_REQUIRE(W && C, "ic_gram_tn: null pointer");
    IC_REQUIRE(M >= 0 && N >= 0 && ldw >= N, "ic_gram_tn: bad size");
    if (N == 0) return IC_OK;
    hipStream_t st = as_stream(stream);
    // C[i][j] and C[j][i] are the same products summed in the same order:
    // the upper triangle on the matrix cores, then mirrored
    GemmArgs g{N, N, M, alpha, 0.0f, W, ldw, 0, W, ldw, 0, C, N, 0, 1, 0, CMASK_UPPER, KR_FULL, 1, PT_OTHER,
               (double)N * (N + 1) * M};
    int rc = gemm_f32(g, st);
    if (rc) return rc;
    return mirror_upper(C, 1, N, N, N * N, st);
}

extern "C" int ic_cholesky(float* H, int64_t batch, int64_t n, int* info, void* workspace, void* stream) {
    IC_REQUIRE(H && info && workspace, "ic_cholesky: null pointer");
    if (n == 0 || batch == 0) return IC_OK;
    hipStream_t st = as_stream(stream);
    IC_CHECK_HIP(hipMemsetAsync(info, 0, batch * sizeof(int), st));
    double* tiles = tiles_at(reinterpret_cast<float*>(workspace) + batch * n * n);
    return potrf(H, batch, n, n, n * n, tiles, info, st);
}

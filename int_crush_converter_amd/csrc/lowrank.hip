// Low-rank eigendecomposition of a symmetric PSD Hessian for the greedy
// search (converter/greedy.py:293-366, _lowrank_decompose).
//
// The reference calls torch.svd_lowrank(H, q = N/2) (falling back to eigh)
// and keeps the eigenpairs above rank_threshold x the largest.  Only the top
// p = min(N, k_cap + oversampling) pairs can ever be used (the greedy
// refuses k > min(512, 0.3 N)), so this builds them by subspace iteration:
//
//   lam ~ lambda_max(H)                   16 power steps on a seeded vector
//   Q0 = orth(G)                          G: seeded Gaussian [n, p]
//   Q_{i+1} = orth((H + mu I) Q_i)        i < iters, mu = 1e-3 lam
//   T = Q^T H Q  (p x p)   ->   T = V diag(d) V^T  (cyclic Jacobi, fp64)
//   eigenvalues d (descending), eigenvectors Q V
//
// The shift mu keeps (H + mu I) Q of full rank when H is singular (a
// calibration Hessian from few samples) and bounds its condition number by
// ~1e3 without changing the eigenvectors; it slows the separation of an
// eigenvalue above the cut (>= 1e-2 lam) from one below by < 10 %.
// orth() is shifted CholeskyQR3: three passes of Y <- Y chol(Y^T Y + s I)^-T,
// the first with s = 1e-5 tr(Y^T Y), which divides the condition number by
// ~1/sqrt(s) so that the two plain passes see <= 76 (mu = 1e-3 lambda_max)
// and fp32 Gram matrices keep them accurate; steps whose basis only feeds the next one
// leave out the third.  Every piece is an fp32-MFMA GEMM or the
// blocked Cholesky / triangular inverse of chol.hip.
//
// The p x p eigenproblem is two-sided cyclic Jacobi in fp64 by blocks of 32
// (below).  Sweeps run until the off-diagonal norm is below 1e-12 of the
// diagonal's, or 40 sweeps.
#include <algorithm>

#include "chol.hpp"

namespace icq {

// ------------------------------------------------------------ helpers

__device__ __forceinline__ uint64_t mix64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

// Standard normal samples from a counter-based hash (Box-Muller).
__global__ void randn_kernel(float* Y, int64_t n, uint64_t seed) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t h = mix64(seed ^ mix64((uint64_t)i));
        const double u1 = ((double)(h >> 11) + 0.5) * 0x1p-53;
        const double u2 = (double)(mix64(h) >> 11) * 0x1p-53;
        Y[i] = (float)(sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2));
    }
}

// y = H x, one wave per row (fp32 products, fp64 sum)
__global__ void matvec_kernel(const float* H, int64_t n, const float* x, float* y) {
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= n) return;
    const int lane = threadIdx.x & 63;
    double acc = 0.0;
    for (int64_t j = lane; j < n; j += 64) acc += (double)(H[row * n + j] * x[j]);
    acc = wave_sum(acc);
    if (lane == 0) y[row] = (float)acc;
}

// x = y / ||y||, out[0] = rel * ||y||  (one work-group; ||y|| = 0 leaves x)
__global__ void normalize_kernel(const float* y, float* x, int64_t n, double rel, double* out) {
    __shared__ double red[4];
    double acc = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) acc += (double)y[i] * (double)y[i];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    const double nrm = sqrt(red[0] + red[1] + red[2] + red[3]);
    if (nrm > 0.0)
        for (int64_t i = threadIdx.x; i < n; i += blockDim.x) x[i] = (float)((double)y[i] / nrm);
    if (threadIdx.x == 0) out[0] = rel * nrm;
}

// part[b] = sum of squares over the block's grid-stride share (fp64)
__global__ void sumsq_kernel(const float* x, int64_t n, double* part) {
    __shared__ double red[4];
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const double v = x[i];
        acc += v * v;
    }
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// T[i][i] -= rel * sqrt(sum part[0..n))  (one work-group of 256; fixed order)
__global__ void sub_frob_diag_kernel(float* T, int64_t p, const double* part, int n, double rel) {
    __shared__ double red[4];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) acc += part[i];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    const double shift = rel * sqrt(red[0] + red[1] + red[2] + red[3]);
    for (int64_t i = threadIdx.x; i < p; i += blockDim.x) T[i * p + i] = (float)((double)T[i * p + i] - shift);
}

// Y += mu * Q  (mu read from device memory)
__global__ void axpy_dev_kernel(float* Y, const float* Q, int64_t n, const double* mu) {
    const float m = (float)mu[0];
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        Y[i] = Y[i] + m * Q[i];
}

// G[i][i] += rel * trace(G)  (one work-group)
__global__ void shift_diag_kernel(float* G, int64_t p, float rel) {
    __shared__ float red[4];
    float acc = 0.0f;
    for (int64_t i = threadIdx.x; i < p; i += blockDim.x) acc += G[i * p + i];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    const float s = rel * (red[0] + red[1] + red[2] + red[3]);
    for (int64_t i = threadIdx.x; i < p; i += blockDim.x) G[i * p + i] = G[i * p + i] + s;
}

// Zero the strict upper triangle of a p x p matrix.
__global__ void zero_upper_kernel(float* X, int64_t p) {
    const int64_t n = p * p;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = idx / p, j = idx - i * p;
        if (j > i) X[idx] = 0.0f;
    }
}

// ------------------------------------------------------------ Jacobi
//
// The p indices (padded to P, a multiple of 64, with zero rows) are taken in
// blocks of 32; a round pairs the blocks (round-robin), each pair's 64 x 64
// part of A is rotated in LDS by one work-group (jacobi_solve_kernel), which
// also collects the product U of its rotations, and the rest of A and V
// follow as fp64 MFMA products with the U (jacobi_apply_kernel).  A sweep
// meets every pair of indices once: the first round also rotates inside the
// blocks.  Latency-bound: the 32 rounds of rotations inside a launch are the
// chain, 1.1 us each (their angle, then LDS traffic: 64 rows of A and of U
// read and written).  For p = 576 a round takes 40 us to solve and 9.4 us to
// apply, 17 rounds a sweep, 6.7 ms in 8 sweeps; a launch per round of p / 2
// single rotations, each over all of A and V, took 8.5 us: 4600 of them, 39
// ms, in as many sweeps.

typedef double doublex4 __attribute__((ext_vector_type(4)));
constexpr int JB = 32, JP = 2 * JB;        // block and pair of blocks
constexpr int JPITCH = JP + 1;             // pitch of a 64-column tile in LDS (doubles): rows and columns
                                           // both spread over the banks

// A = fp64((T + T^T) / 2) and V = I, padded to P x P: zeros and the identity.
__global__ void jacobi_init_kernel(const float* T, int64_t p, int64_t P, double* A, double* V) {
    const int64_t n = P * P;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = idx / P, j = idx - i * P;
        A[idx] = i < p && j < p ? 0.5 * ((double)T[i * p + j] + (double)T[j * p + i]) : 0.0;
        V[idx] = i == j ? 1.0 : 0.0;
    }
}

// Pair k of round r (round-robin over n items, n even): item n - 1 meets r,
// the others meet by reflection about r.  Returned ordered (a < b).
__device__ __forceinline__ void jpair(int k, int r, int n, int& a, int& b) {
    const int m = n - 1;
    if (k == 0) {
        a = r;
        b = m;
    } else {
        a = r + k;
        if (a >= m) a -= m;
        b = r - k;
        if (b < 0) b += m;
    }
    if (a > b) {
        const int t = a;
        a = b;
        b = t;
    }
}

// Row of the matrix that index i (0 .. 63) of the pair of blocks (I, J) is.
__device__ __forceinline__ int jrow(int i, int I, int J) { return i < JB ? I * JB + i : J * JB + i - JB; }

// 1 / x and 1 / sqrt(x) from the hardware estimates: two Newton steps to the
// last bits of fp64 (half the dependent operations of the IEEE quotient and
// root; the rotations are a serial chain).
__device__ __forceinline__ double rcp64(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}
__device__ __forceinline__ double rsq64(double x) {
    const double h = -0.5 * x;
    double r = __builtin_amdgcn_rsq(x);
    r = r * fma(h * r, r, 1.5);
    return r * fma(h * r, r, 1.5);
}

// Rotation annihilating apq (Golub & Van Loan, symmetric Schur 2x2):
// J = [[c, s], [-s, c]] on (p, q), A' = J^T A J; t = tan, the smaller root
// 2 apq / (d + sign(d) sqrt(d^2 + 4 apq^2)) of t^2 + (d / apq) t - 1 = 0,
// d = aqq - app.  Below 1e-140 (the squares underflow) apq counts as zero.
__device__ __forceinline__ void jrot(double app, double apq, double aqq, double& c, double& s, double& t) {
    const double d = aqq - app, w = fma(d, d, 4.0 * apq * apq);
    if (fabs(apq) < 1e-140) {
        c = 1.0;
        s = 0.0;
        t = 0.0;
        return;
    }
    const double den = fabs(d) + w * rsq64(w);
    t = 2.0 * apq * rcp64(den);
    if (d < 0.0) t = -t;
    c = rsq64(fma(t, t, 1.0));
    s = t * c;
}

// Pair blockIdx.x of round r: its 64 x 64 part of Ain through all rotations
// between its two blocks (full: and inside them) to Aout, and their product
// to U[pair] (64 x 64).  Per round of 32 disjoint rotations: their angles
// (32 threads), then the 2 x 2 blocks of pairs P < C (mirrored, so that A
// stays exactly symmetric), the diagonal ones and U's columns.
__global__ __launch_bounds__(1024) void jacobi_solve_kernel(const double* Ain, double* Aout, double* U, int64_t P,
                                                           int r, int nblk, int full) {
    __shared__ double A[JP][JPITCH], W[JP][JPITCH];
    __shared__ double rc[JB], rs[JB], rt[JB];
    const int t = threadIdx.x;
    int I, J;
    jpair(blockIdx.x, r, nblk, I, J);
    double a0[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = (t >> 6) + 16 * u, j = t & 63;
        a0[u] = Ain[(int64_t)jrow(i, I, J) * P + jrow(j, I, J)];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = (t >> 6) + 16 * u, j = t & 63;
        A[i][j] = a0[u];
        W[i][j] = i == j ? 1.0 : 0.0;
    }
    // this thread's 2 x 2 block of pairs pr < pc (t < 496)
    int pr = 0, pc = 0;
    {
        int id = t;
        while (pr < JB - 1 && id >= JB - 1 - pr) { id -= JB - 1 - pr; ++pr; }
        pc = pr + 1 + id;
    }
    __syncthreads();
    const int rounds = full ? JP - 1 : JB;
    for (int q = 0; q < rounds; ++q) {
        auto pair_of = [&](int k, int& a, int& b) {
            if (full) {
                jpair(k, q, JP, a, b);
            } else {
                a = k;
                b = JB + ((k + q) & (JB - 1));
            }
        };
        if (t < JB) {
            int a, b;
            pair_of(t, a, b);
            jrot(A[a][a], A[a][b], A[b][b], rc[t], rs[t], rt[t]);
        }
        __syncthreads();
        if (t < JB * (JB - 1) / 2) {
            int a, b, c, d;
            pair_of(pr, a, b);
            pair_of(pc, c, d);
            const double cp = rc[pr], sp = rs[pr], cc = rc[pc], sc = rs[pc];
            const double x00 = A[a][c], x01 = A[a][d], x10 = A[b][c], x11 = A[b][d];
            const double y00 = cp * x00 - sp * x10, y01 = cp * x01 - sp * x11;
            const double y10 = sp * x00 + cp * x10, y11 = sp * x01 + cp * x11;
            const double z00 = cc * y00 - sc * y01, z01 = sc * y00 + cc * y01;
            const double z10 = cc * y10 - sc * y11, z11 = sc * y10 + cc * y11;
            A[a][c] = A[c][a] = z00;
            A[a][d] = A[d][a] = z01;
            A[b][c] = A[c][b] = z10;
            A[b][d] = A[d][b] = z11;
        } else if (t >= 512 && t < 512 + JB) {
            int a, b;
            pair_of(t - 512, a, b);
            const double apq = A[a][b], tp = rt[t - 512];
            A[a][a] = A[a][a] - tp * apq;
            A[b][b] = A[b][b] + tp * apq;
            A[a][b] = A[b][a] = 0.0;
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int row = (t >> 5) + 32 * u, k = t & 31;
            int a, b;
            pair_of(k, a, b);
            const double c = rc[k], s = rs[k], va = W[row][a], vb = W[row][b];
            W[row][a] = c * va - s * vb;
            W[row][b] = s * va + c * vb;
        }
        __syncthreads();
    }
    double* Up = U + (int64_t)blockIdx.x * JP * JP;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int idx = t + 1024 * u, i = idx / JP, j = idx % JP;
        Aout[(int64_t)jrow(i, I, J) * P + jrow(j, I, J)] = A[i][j];
        Up[idx] = W[i][j];
    }
}

// D += A^T-or-A times B for this wave's 16 x 32 part (rows r0, columns c0) of
// a 32 x 64 product with K = 64: a(k, i) and b(k, j) read the operands in LDS.
// v_mfma_f64_16x16x4_f64: A[i = l%16][k = l/16], B[k = l/16][j = l%16],
// D[i = l/16 + 4 v][j = l%16].
template <typename FA, typename FB>
__device__ __forceinline__ void jmul(doublex4 (&acc)[2], FA&& a, FB&& b, int r0, int c0, int lane) {
    const int li = lane & 15, lk = lane >> 4;
    acc[0] = acc[1] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k0 = 0; k0 < JP; k0 += 4) {
        const double av = a(k0 + lk, r0 + li);
#pragma unroll
        for (int c = 0; c < 2; ++c)
            acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, b(k0 + lk, c0 + 16 * c + li), acc[c], 0, 0, 0);
    }
}

// The rest of round r: for pairs of blocks x < y the part A[x][y] becomes
// U_x^T A[x][y] U_y (and its mirror), and 64 rows of V times each pair's
// columns V U.  Work-group: 32 rows of one such part (a pair's part on the
// diagonal comes from jacobi_solve_kernel).  Blocks [0, 2 np (np - 1) / 2):
// A; then 2 np^2: V (in place: a work-group reads only what it writes).
__global__ __launch_bounds__(256) void jacobi_apply_kernel(const double* Ain, double* Aout, double* V, const double* U,
                                                          int64_t P, int r, int nblk) {
    __shared__ double S[JP][JPITCH], Ux[JP][JB + 2], Uy[JP][JPITCH], Y[JB][JPITCH];
    const int np = nblk / 2, t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int li = lane & 15, lk = lane >> 4, r0 = (wave >> 1) * 16, c0 = (wave & 1) * 32;
    const int nA = np * (np - 1);
    const int id = blockIdx.x;
    const bool isA = id < nA;
    int x, y, h;
    if (isA) {
        int k = id >> 1;
        h = id & 1;
        x = 0;
        while (k >= np - 1 - x) { k -= np - 1 - x; ++x; }
        y = x + 1 + k;
    } else {
        h = (id - nA) & 1;
        x = ((id - nA) >> 1) / np;
        y = ((id - nA) >> 1) - x * np;
    }
    int I, J, K = 0, L = 0;
    jpair(y, r, nblk, I, J);
    if (isA) jpair(x, r, nblk, K, L);
    // all loads in flight before the first LDS store
    const double* Uyp = U + (int64_t)y * JP * JP;
    double uy[16], ux[8], sv[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) uy[u] = Uyp[t + 256 * u];
    doublex4 acc[2];
    if (isA) {
        const double* Uxp = U + (int64_t)x * JP * JP;
#pragma unroll
        for (int u = 0; u < 16; ++u)
            sv[u] = Ain[(int64_t)jrow((t >> 6) + 4 * u, K, L) * P + jrow(t & 63, I, J)];
#pragma unroll
        for (int u = 0; u < 8; ++u) ux[u] = Uxp[((t >> 5) + 8 * u) * JP + h * JB + (t & 31)];
#pragma unroll
        for (int u = 0; u < 16; ++u) S[(t >> 6) + 4 * u][t & 63] = sv[u];
#pragma unroll
        for (int u = 0; u < 8; ++u) Ux[(t >> 5) + 8 * u][t & 31] = ux[u];
    } else {
#pragma unroll
        for (int u = 0; u < 8; ++u)
            sv[u] = V[((int64_t)x * JP + h * JB + (t >> 6) + 4 * u) * P + jrow(t & 63, I, J)];
#pragma unroll
        for (int u = 0; u < 8; ++u) Y[(t >> 6) + 4 * u][t & 63] = sv[u];
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) Uy[(t >> 6) + 4 * u][t & 63] = uy[u];
    if (isA) {
        __syncthreads();
        jmul(acc, [&](int k, int i) { return Ux[k][i]; }, [&](int k, int j) { return S[k][j]; }, r0, c0, lane);
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int v = 0; v < 4; ++v) Y[r0 + lk + 4 * v][c0 + 16 * c + li] = acc[c][v];
    }
    __syncthreads();
    jmul(acc, [&](int k, int i) { return Y[i][k]; }, [&](int k, int j) { return Uy[k][j]; }, r0, c0, lane);
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = r0 + lk + 4 * v, col = jrow(c0 + 16 * c + li, I, J);
            if (isA) {
                const int row = jrow(h * JB + i, K, L);
                Aout[(int64_t)row * P + col] = acc[c][v];
                Aout[(int64_t)col * P + row] = acc[c][v];
            } else {
                V[((int64_t)x * JP + h * JB + i) * P + col] = acc[c][v];
            }
        }
}

// part[2 b] = off-diagonal sum of squares, part[2 b + 1] = diagonal's.
__global__ void offdiag_kernel(const double* A, int64_t p, double* part) {
    __shared__ double red[2][4];
    double off = 0.0, dia = 0.0;
    const int64_t n = p * p;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = idx / p, j = idx - i * p;
        const double v = A[idx];
        if (i == j) dia += v * v;
        else off += v * v;
    }
    off = wave_sum(off);
    dia = wave_sum(dia);
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = off;
        red[1][threadIdx.x >> 6] = dia;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = red[0][0] + red[0][1] + red[0][2] + red[0][3];
        part[2 * blockIdx.x + 1] = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    }
}

// out[0], out[1] = the sums of the pairs (one work-group of 256; fixed order)
__global__ void finish_pairs_kernel(const double* part, int n, double* out) {
    __shared__ double red[2][4];
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) {
        a += part[2 * i];
        b += part[2 * i + 1];
    }
    a = wave_sum(a);
    b = wave_sum(b);
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = a;
        red[1][threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        out[0] = red[0][0] + red[0][1] + red[0][2] + red[0][3];
        out[1] = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    }
}

// Descending order of the first p diagonal entries of A (pitch P; ties:
// lower index first): eigenvalue j goes to position rank[j].
__global__ __launch_bounds__(256) void ritz_rank_kernel(const double* A, int64_t p, int64_t P, float* evals,
                                                       int* rank) {
    __shared__ double d[256];
    const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const double dj = j < p ? A[j * P + j] : 0.0;
    int r = 0;
    for (int64_t i0 = 0; i0 < p; i0 += 256) {
        __syncthreads();
        if (i0 + threadIdx.x < p) d[threadIdx.x] = A[(i0 + threadIdx.x) * P + i0 + threadIdx.x];
        __syncthreads();
        const int m = (int)std::min<int64_t>(256, p - i0);
        for (int i = 0; i < m; ++i) r += (d[i] > dj || (d[i] == dj && i0 + i < j)) ? 1 : 0;
    }
    if (j < p) {
        evals[r] = (float)dj;
        rank[j] = r;
    }
}

// Vs[i][rank[j]] = V[i][j], p x p (a work-group per row)
__global__ void ritz_columns_kernel(const double* V, const int* rank, int64_t p, int64_t P, float* Vs) {
    for (int64_t j = threadIdx.x; j < p; j += blockDim.x)
        Vs[blockIdx.x * p + rank[j]] = (float)V[blockIdx.x * P + j];
}

static int egrid_lr(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(cdiv(n, 256), 4096)); }

static size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// Workspace carve-up (every piece 256-byte aligned).
struct LrWork {
    float *Y, *Q, *G, *X, *T, *Vs, *x, *y, *Gp;
    double *tiles, *A0, *A1, *V, *U, *part, *scal;
    int *info, *rank;
};

constexpr int LR_PARTS = 1024;   // partial sums of the reductions
constexpr int GRAM_SPLIT = 8;    // K chunks of the p x p Gram matrices (K = n)

static size_t lr_layout(int64_t n, int64_t p, char* base, LrWork* w) {
    size_t off = 0;
    auto take = [&](size_t bytes) {
        char* ptr = base ? base + off : nullptr;
        off += align256(bytes);
        return ptr;
    };
    const size_t P = (size_t)cdiv(p, JP) * JP;   // Jacobi's padded order
    const size_t np4 = (size_t)n * p * 4, pp4 = (size_t)p * p * 4, pp8 = P * P * 8;
    LrWork t{};
    t.Y = (float*)take(np4);
    t.Q = (float*)take(np4);
    t.G = (float*)take(pp4);
    t.X = (float*)take(pp4);
    t.T = (float*)take(pp4);
    t.Vs = (float*)take(pp4);
    t.x = (float*)take((size_t)n * 4);
    t.Gp = (float*)take((size_t)GRAM_SPLIT * pp4);
    t.y = (float*)take((size_t)n * 4);
    t.tiles = (double*)take((size_t)tile_doubles(1, p) * 8);
    t.A0 = (double*)take(pp8);
    t.A1 = (double*)take(pp8);
    t.V = (double*)take(pp8);
    t.U = (double*)take(P / JP * JP * JP * 8);
    t.rank = (int*)take((size_t)p * 4);
    t.part = (double*)take((size_t)LR_PARTS * 2 * 8);
    t.scal = (double*)take(8 * 8);
    t.info = (int*)take(64);
    if (base) *w = t;
    return off + 256;
}

// G[i][j] = sum over the S partials (fixed order), lower triangle
__global__ void sum_partials_kernel(const float* Gp, int S, int64_t pp, float* G) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < pp; i += (int64_t)gridDim.x * blockDim.x) {
        float acc = Gp[i];
        for (int s = 1; s < S; ++s) acc = acc + Gp[s * pp + i];
        G[i] = acc;
    }
}

// G = A^T B (p x p, part `cmask`; A, B [n, p]) with K = n cut into up to
// GRAM_SPLIT chunks of a batched GEMM: the p x p output alone has too few
// tiles to fill the chip.
static int gram(const float* A, const float* B, int64_t n, int64_t p, float* G, const LrWork& w, int cmask,
                hipStream_t st) {
    const int64_t kc = cdiv(cdiv(n, GRAM_SPLIT), 32) * 32;
    const int S = (int)cdiv(n, kc);
    const int64_t pp = p * p;
    int rc;
    if (S > 1) {
        GemmArgs g{p, p, kc, 1.0f, 0.0f, A, p, kc * p, B, p, kc * p, w.Gp, p, pp, 1, 0, cmask, KR_FULL, S - 1,
                   PT_OTHER};
        if ((rc = gemm_f32(g, st))) return rc;
    }
    const int64_t k0 = (S - 1) * kc;
    GemmArgs g{p, p, n - k0, 1.0f, 0.0f, A + k0 * p, p, 0, B + k0 * p, p, 0, w.Gp + (S - 1) * pp, p, 0, 1, 0, cmask,
               KR_FULL, 1, PT_OTHER};
    if ((rc = gemm_f32(g, st))) return rc;
    hipLaunchKernelGGL(sum_partials_kernel, dim3(egrid_lr(pp)), dim3(256), 0, st, w.Gp, S, pp, G);
    IC_CHECK_LAUNCH();
    return IC_OK;
}

// One CholeskyQR pass: Q = Y R^-1 with R^T R = Y^T Y + shift_rel tr(Y^T Y) I.
static int cholqr_pass(const float* Y, float* Q, int64_t n, int64_t p, float shift_rel, const LrWork& w,
                       hipStream_t st) {
    int rc = gram(Y, Y, n, p, w.G, w, CMASK_LOWER, st);
    if (rc) return rc;
    if (shift_rel > 0.0f) {
        hipLaunchKernelGGL(shift_diag_kernel, dim3(1), dim3(256), 0, st, w.G, p, shift_rel);
        IC_CHECK_LAUNCH();
    }
    if ((rc = potrf(w.G, 1, p, p, p * p, w.tiles, w.info, st))) return rc;
    if ((rc = trtri(w.G, w.X, 1, p, p, p * p, w.tiles, st))) return rc;
    hipLaunchKernelGGL(zero_upper_kernel, dim3(egrid_lr(p * p)), dim3(256), 0, st, w.X, p);
    IC_CHECK_LAUNCH();
    // Q = Y X^T  (X = L^-1 lower, so op(B) = X^T is upper triangular)
    GemmArgs q{n, p, p, 1.0f, 0.0f, Y, p, 0, w.X, p, 0, Q, p, 0, 0, 1, CMASK_FULL, KR_FULL, 1, PT_OTHER};
    return gemm_f32(q, st);
}

// Orthonormal basis of the columns of w.Y into w.Q (the two buffers trade
// places as needed; Y's content is lost).  ORTH_START: a Gaussian start
// (cond ~ (1 + sqrt(p/n)) / (1 - sqrt(p/n))), two plain passes.  ORTH_FULL:
// shifted CholeskyQR3.  ORTH_STEP: its first two passes, after which the next
// product with (H + mu I) has a well-conditioned basis of the same space.
// (H + mu I) Q has a condition number of 1 / mu = 1e3 at most; the shift,
// 1e-5 of a trace of up to p times the largest, leaves sqrt(1e-5 p) 1e3 = 76
// at p = 576, and the second pass an error of about 2^-24 76^2 = 4e-4.  Seen
// over six Hessians (p 244-576; log-normal, log-spaced, 40 eigenvalues above
// zeros): 12 and 3e-5 at most, 2 and 4e-6 as a rule.
enum Orth { ORTH_START, ORTH_STEP, ORTH_FULL };
static int orth(LrWork& w, int64_t n, int64_t p, Orth kind, hipStream_t st) {
    for (int pass = 0; pass < (kind == ORTH_FULL ? 3 : 2); ++pass) {
        if (pass) std::swap(w.Y, w.Q);
        int rc = cholqr_pass(w.Y, w.Q, n, p, pass == 0 && kind != ORTH_START ? 1e-5f : 0.0f, w, st);
        if (rc) return rc;
    }
    return IC_OK;
}

constexpr int JACOBI_MAX_SWEEPS = 40;

}  // namespace icq

using namespace icq;

extern "C" int64_t ic_lowrank_workspace_bytes(int64_t n, int64_t p) {
    if (n <= 0 || p <= 0) return 256;
    return (int64_t)lr_layout(n, p, nullptr, nullptr);
}

extern "C" int ic_lowrank_eigs(const float* H, int64_t n, int64_t p, int iters, unsigned long long seed,
                               float refuse_rel, float* evals, float* evecs, int* sweeps_out, void* workspace,
                               void* stream) {
    IC_REQUIRE(H && evals && evecs && workspace, "ic_lowrank_eigs: null pointer");
    IC_REQUIRE(n >= 2 && p >= 2 && p <= n && p % 2 == 0, "ic_lowrank_eigs: need 2 <= p <= n, p even");
    IC_REQUIRE(p <= 4096 && iters >= 0 && iters <= 64, "ic_lowrank_eigs: p <= 4096, 0 <= iters <= 64");
    IC_REQUIRE(refuse_rel >= 0.0f, "ic_lowrank_eigs: refuse_rel must be >= 0");
    hipStream_t st = as_stream(stream);
    LrWork w;
    char* base = reinterpret_cast<char*>((reinterpret_cast<uintptr_t>(workspace) + 255) & ~(uintptr_t)255);
    lr_layout(n, p, base, &w);
    // info[0]: the orthonormalisations; info[1 + i]: the certificate's i-th test
    // (a factorisation reports a bad pivot only where none is reported yet)
    IC_CHECK_HIP(hipMemsetAsync(w.info, 0, 3 * sizeof(int), st));
    const int64_t np = n * p;
    // mu = 1e-3 lambda_max estimate (power iteration from a seeded vector)
    constexpr int POWER_STEPS = 16;
    hipLaunchKernelGGL(randn_kernel, dim3(egrid_lr(n)), dim3(256), 0, st, w.y, n, (uint64_t)seed ^ 0x5eedull);
    IC_CHECK_LAUNCH();
    hipLaunchKernelGGL(normalize_kernel, dim3(1), dim3(256), 0, st, w.y, w.x, n, 1e-3, w.scal);
    IC_CHECK_LAUNCH();
    for (int i = 0; i < POWER_STEPS; ++i) {
        hipLaunchKernelGGL(matvec_kernel, dim3((unsigned)cdiv(n, 4)), dim3(256), 0, st, H, n, w.x, w.y);
        IC_CHECK_LAUNCH();
        hipLaunchKernelGGL(normalize_kernel, dim3(1), dim3(256), 0, st, w.y, w.x, n, 1e-3, w.scal);
        IC_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL(randn_kernel, dim3(egrid_lr(np)), dim3(256), 0, st, w.Y, np, (uint64_t)seed);
    IC_CHECK_LAUNCH();
    int rc = orth(w, n, p, ORTH_START, st);
    if (rc) return rc;
    // the refusal certificate is tried after one and after two steps (the
    // random start's Ritz values sit near the mean eigenvalue; one step of
    // (H + mu I) already lifts them for Hessians of high rank)
    const int test_lo = refuse_rel > 0.0f ? std::min(iters, 1) : -1;
    const int test_hi = refuse_rel > 0.0f ? std::min(iters, 2) : -1;
    for (int it = 0;; ++it) {
        // Y = H Q
        GemmArgs g{n, p, n, 1.0f, 0.0f, H, n, 0, w.Q, p, 0, w.Y, p, 0, 0, 0, CMASK_FULL, KR_FULL, 1, PT_OTHER};
        if ((rc = gemm_f32(g, st))) return rc;
        if (it >= test_lo && it <= test_hi && test_lo >= 0) {
            // Refusal certificate: if T - refuse_rel ||H||_F I is positive definite,
            // every Ritz value exceeds refuse_rel ||H||_F >= refuse_rel lambda_max,
            // and by interlacing so do the p largest eigenvalues of H.
            if ((rc = gram(w.Q, w.Y, n, p, w.T, w, CMASK_LOWER, st))) return rc;
            hipLaunchKernelGGL(sumsq_kernel, dim3(LR_PARTS), dim3(256), 0, st, H, n * n, w.part);
            IC_CHECK_LAUNCH();
            hipLaunchKernelGGL(sub_frob_diag_kernel, dim3(1), dim3(256), 0, st, w.T, p, w.part, LR_PARTS,
                               (double)refuse_rel);
            IC_CHECK_LAUNCH();
            int* test_info = w.info + 1 + (it - test_lo);
            if ((rc = potrf(w.T, 1, p, p, p * p, w.tiles, test_info, st))) return rc;
            int pd_info = 0;
            IC_CHECK_HIP(hipMemcpyAsync(&pd_info, test_info, sizeof(int), hipMemcpyDeviceToHost, st));
            IC_CHECK_HIP(hipStreamSynchronize(st));
            if (pd_info == 0) {
                if (sweeps_out) *sweeps_out = 0;
                return IC_LOWRANK_REFUSED;
            }
        }
        if (it == iters) break;
        hipLaunchKernelGGL(axpy_dev_kernel, dim3(egrid_lr(np)), dim3(256), 0, st, w.Y, w.Q, np, w.scal);
        IC_CHECK_LAUNCH();
        // the certificate and the Rayleigh-Ritz step want an orthonormal basis
        const bool full = it + 1 == iters || (it + 1 >= test_lo && it + 1 <= test_hi);
        if ((rc = orth(w, n, p, full ? ORTH_FULL : ORTH_STEP, st))) return rc;
    }
    // Rayleigh-Ritz: T = Q^T (H Q)
    if ((rc = gram(w.Q, w.Y, n, p, w.T, w, CMASK_FULL, st))) return rc;
    int info = 0;
    IC_CHECK_HIP(hipMemcpyAsync(&info, w.info, sizeof(int), hipMemcpyDeviceToHost, st));
    IC_CHECK_HIP(hipStreamSynchronize(st));
    if (info != 0) return fail(IC_ERR_RANGE, "ic_lowrank_eigs: orthonormalisation lost positive definiteness");
    const int64_t P = cdiv(p, JP) * JP;
    const int nblk = (int)(P / JB), npair = nblk / 2;
    hipLaunchKernelGGL(jacobi_init_kernel, dim3(egrid_lr(P * P)), dim3(256), 0, st, w.T, p, P, w.A0, w.V);
    IC_CHECK_LAUNCH();
    double *A = w.A0, *An = w.A1;
    const unsigned apply = (unsigned)(npair * (npair - 1) + 2 * npair * npair);
    const int off_blocks = (int)std::min<int64_t>(LR_PARTS, cdiv(P * P, 256));
    int sweeps = 0;
    for (; sweeps < JACOBI_MAX_SWEEPS; ++sweeps) {
        hipLaunchKernelGGL(offdiag_kernel, dim3(off_blocks), dim3(256), 0, st, A, P, w.part);
        IC_CHECK_LAUNCH();
        hipLaunchKernelGGL(finish_pairs_kernel, dim3(1), dim3(256), 0, st, w.part, off_blocks, w.scal + 2);
        IC_CHECK_LAUNCH();
        double od[2];
        IC_CHECK_HIP(hipMemcpyAsync(od, w.scal + 2, sizeof(od), hipMemcpyDeviceToHost, st));
        IC_CHECK_HIP(hipStreamSynchronize(st));
        if (!(od[0] > 1e-24 * od[1])) break;   // converged (or NaN: the caller sees NaN eigenvalues)
        for (int r = 0; r < nblk - 1; ++r) {
            hipLaunchKernelGGL(jacobi_solve_kernel, dim3(npair), dim3(1024), 0, st, A, An, w.U, P, r, nblk,
                               r == 0 ? 1 : 0);
            IC_CHECK_LAUNCH();
            hipLaunchKernelGGL(jacobi_apply_kernel, dim3(apply), dim3(256), 0, st, A, An, w.V, w.U, P, r, nblk);
            IC_CHECK_LAUNCH();
            std::swap(A, An);
        }
    }
    if (sweeps_out) *sweeps_out = sweeps;
    hipLaunchKernelGGL(ritz_rank_kernel, dim3((unsigned)cdiv(p, 256)), dim3(256), 0, st, A, p, P, evals, w.rank);
    IC_CHECK_LAUNCH();
    hipLaunchKernelGGL(ritz_columns_kernel, dim3((unsigned)p), dim3(256), 0, st, w.V, w.rank, p, P, w.Vs);
    IC_CHECK_LAUNCH();
    // eigenvectors of H: Q Vs
    GemmArgs e{n, p, p, 1.0f, 0.0f, w.Q, p, 0, w.Vs, p, 0, evecs, p, 0, 0, 0, CMASK_FULL, KR_FULL, 1, PT_OTHER};
    return gemm_f32(e, st);
}

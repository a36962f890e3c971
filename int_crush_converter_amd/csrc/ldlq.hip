// LDLQ helpers (per-element scales, iteration MSE, scale refinement,
// least-squares row scales) and the full-rank greedy coordinate descent.
//
// Greedy (converter/greedy.py:487-541): for every column j, every row picks
// the grid value minimising (e+d)^2 H_jj + 2 (e+d) cross, cross =
// err . H[j, :] - e_j H_jj.  Columns are processed in blocks of 64: one
// fp32-MFMA GEMM gives err @ H[blk, :]^T for the whole block at its start,
// and the changes d_j' of earlier columns of the block are added exactly as
// sum_j' d_j' H[j', j] - the same quantity in exact arithmetic as the
// reference's per-column GEMV (its fp32 rounding differs).
#include "gemm_dev.hpp"
#include "split.hpp"
#include "torchsum.hpp"

namespace icq {

constexpr int GB = 64;          // greedy column block
constexpr int GQ = 4;           // lanes per row in the greedy block kernel
constexpr int64_t GSB = 512;    // greedy super-block (columns)

__device__ __forceinline__ float nclampmin(float x, float lo) { return x != x ? x : (x < lo ? lo : x); }

// s_r = max(absmax_r / div, 1e-5) (no upper clamp, ldlq.py:212); S = broadcast
__global__ void ldlq_init_scales_kernel(const float* ramax, int64_t rows, int64_t cols, float div, float* srow,
                                        float* S) {
    const int64_t total = rows * cols;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / cols;
        const float s = nclampmin(ramax[r] / div, 1e-5f);
        S[i] = s;
        if (i - r * cols == 0 && srow) srow[r] = s;
    }
}

// Non-finite scales -> nan_to_num(nan=1e-8, posinf=1e30, neginf=1e-8).clamp(min=1e-8)
__global__ void sanitize_scales_kernel(float* S, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        float v = S[i];
        if (v != v) v = 1e-8f;
        else if (isinf(v)) v = v > 0 ? 1e30f : 1e-8f;
        S[i] = v < 1e-8f ? 1e-8f : v;
    }
}

// partial sums of (W - Q*S)^2 in fp64 (product and difference in fp32)
__global__ __launch_bounds__(256) void ldlq_mse_kernel(const float* W, const int8_t* Q, const float* S, int64_t n,
                                                       double* part) {
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        float d = W[i] - (float)Q[i] * S[i];
        acc += (double)d * (double)d;
    }
    __shared__ double sh[4];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

__global__ __launch_bounds__(256) void sum_parts_kernel(const double* part, int n, double* out) {
    double a = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) a += part[i];
    __shared__ double sh[4];
    a = wave_sum(a);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = a;
    __syncthreads();
    if (threadIdx.x == 0) *out = (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

// converter/ldlq.py:553-599
__global__ void ldlq_update_kernel(const float* W, const int8_t* Q, const float* cur, const float* flat, int64_t n,
                                   float momentum, float lo, float hi, float* out) {
    const float keep = 1.0f - momentum;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float w = W[i], q = (float)Q[i];
        const bool nonzero = q != 0.0f;
        const bool consistent = fabsf(w) > 1e-8f && (w * q) > 0.0f;
        float v = cur[i];
        if (nonzero && consistent) {
            float comp = clampf(fabsf(w) / fabsf(q), lo, hi);
            v = momentum > 0.0f ? momentum * cur[i] + keep * comp : comp;
        } else if (nonzero) {
            v = clampf(flat[i], lo, hi);
        }
        out[i] = v;
    }
}

// Per-row least squares scale clamp(sum(q w) / max(sum(q q), 1e-8), min=1e-5)
// (ldlq.py:227-231, 262-265).  The reference sums the fp32 products
// (Q_float * W, Q_float * Q_float) over each row with torch's CPU inner
// sum (one CPU thread per row when there is more than one row), so the
// sums here follow that order: lane s (< 32) of a row's wave takes
// sequence s of the numerator, lane 32 + s that of the denominator, and one
// lane per sum finishes it (the leftover vectors, the merge, the leftover
// scalars, the lanes).  A wave per row, four rows per work-group.
__global__ __launch_bounds__(256) void ls_scales_kernel(const int8_t* Q, const float* W, int64_t rows, int64_t cols,
                                                        float* out) {
    __shared__ float part[4][2][SUM_SEQ];
    __shared__ float dens[4];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t r0 = (int64_t)blockIdx.x * 4 + wv;
    const bool live = r0 < rows;
    const int64_t r = live ? r0 : rows - 1;
    const int8_t* q = Q + r * cols;
    const float* w = W + r * cols;
    auto xn = [&](int64_t i) { const float qf = (float)q[i]; return qf * w[i]; };
    auto xd = [&](int64_t i) { const float qf = (float)q[i]; return qf * qf; };
    const int which = lane >> 5, s = lane & (SUM_SEQ - 1);
    float sum = 0.0f;
    if (cols >= SUM_VEC) {
        const int64_t n4 = cols / SUM_VEC / 4;
        const int lp = cascade_lp(n4);
        part[wv][which][s] = which == 0 ? cascade_seq([&](int64_t m) { return xn(m * SUM_SEQ + s); }, n4, lp)
                                        : cascade_seq([&](int64_t m) { return xd(m * SUM_SEQ + s); }, n4, lp);
        __syncthreads();
        if (s == 0) sum = which == 0 ? inner_sum_finish(part[wv][0], xn, cols) : inner_sum_finish(part[wv][1], xd, cols);
    } else {
        __syncthreads();
        if (s == 0) sum = which == 0 ? inner_sum_short(xn, cols) : inner_sum_short(xd, cols);
    }
    if (lane == 32) dens[wv] = sum;
    __syncthreads();
    if (lane == 0 && live) {
        float d32 = dens[wv];
        d32 = d32 < 1e-8f ? 1e-8f : d32;
        out[r] = nclampmin(sum / d32, 1e-5f);
    }
}

// err = Q * S - W with S per row (pe 0: sc[rows], the least-squares row
// scales the pipeline passes) or per element (pe 1: sc[rows, cols])
__global__ void greedy_err_kernel(const int8_t* Q, const float* sc, int pe, const float* W, int64_t rows,
                                  int64_t cols, float* err, float* Qf) {
    const int64_t total = rows * cols;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const float q = (float)Q[i];
        Qf[i] = q;
        err[i] = q * sc[pe ? i : i / cols] - W[i];
    }
}

// A 64-column block of a greedy pass for GQR rows is run by one wave, GQ = 4
// lanes (a DPP quad) per row.  Lane p of a row owns the block columns
// j = 4 m + p (m = 0..15) and keeps, in registers, their err, code and cross
// term
//   c_j = err @ H[:, j] as of the start of the block
//         + sum over the block columns j' < j decided so far of
//           (err_new - err_old)_j' * H[j', j],
// the changes added one column at a time in the column order (the rank-1
// corrections of converter/greedy.py:255-258, as fused multiply-adds).
// Column jl's decision (converter/greedy.py:80-95: the grid value with the
// least (e + d)^2 H_jj + 2 (e + d) cross, cross = c_j - e H_jj, the first
// one on a tie) is made by its owner from the two grid values around the
// continuous minimiser t = q - (cross / H_jj + e) / s: the cost is a convex
// quadratic in the grid value, so when its fp32 rounding is small against
// the gap H_jj s^2 between neighbouring grid values (|cross| <= 128 H_jj s,
// |t| < 2^16, H_jj and s^2 in a normal range) no other grid value can tie or
// beat the better of the two, and the full scan's answer is that one.
// Otherwise the whole grid is scanned in increasing order, as the reference
// does.  The change is then broadcast over the quad and every lane adds its
// products to the cross terms of its later columns.  H is the matrix of the
// cross terms (the Hessian, or its low-rank truncation) and hd its exact
// diagonal H_jj (null: the diagonal of H).
constexpr int GQR = 64 / GQ;      // rows per work-group
constexpr int GSLOT = GB / GQ;    // block columns per lane
constexpr float GREEDY_GAMMA = 128.0f;
constexpr float GREEDY_TMAX = 65536.0f;

// The reference's scan over the whole grid (first minimum, codes start at
// q): {code, new err}.
__device__ __forceinline__ float2 greedy_scan(float e, float q, float s, float h, float cross, float qmin,
                                              float qmax) {
    float best = 1e30f, bq = q;
    for (float g = qmin; g <= qmax; g += 1.0f) {
        const float ne = e + (g - q) * s;
        const float cost = ne * ne * h + 2.0f * ne * cross;
        if (cost < best) {
            best = cost;
            bq = g;
        }
    }
    bq = clampf(bq, qmin, qmax);
    return make_float2(bq, e + (bq - q) * s);
}

// The guard scale of greedy_decide: GREEDY_GAMMA s, or NaN for a scale
// outside the window's domain.
__device__ __forceinline__ float greedy_guard(float s) {
    const float s2 = s * s;
    return (s > 0.0f && s2 >= 0x1p-40f && s2 <= 0x1p30f) ? GREEDY_GAMMA * s : __builtin_nanf("");
}

// The window decision for one column of one row: err e, code q, running
// cross-term sum c (before the diagonal term), column data cv = {H_jj,
// H_jj or NaN, 1 / H_jj}, the scale s of this element, 1 / s and the guard
// scale sg = greedy_guard(s).  {code, new err}; fast: the window's answer is
// the full scan's.
__device__ __forceinline__ float2 greedy_decide(float e, float q, float c, float4 cv, float s, float is, float sg,
                                                float qmin, float qmax, bool& fast) {
    const float h = cv.x;
    const float cross = c - e * h;
    const float tt = q - fmaf(cross, cv.z, e) * is;
    const float g0 = __builtin_amdgcn_fmed3f(floorf(tt), qmin, qmax - 1.0f), g1 = g0 + 1.0f;
    const float n0 = e + (g0 - q) * s, n1 = e + (g1 - q) * s;
    const float c0 = n0 * n0 * h + 2.0f * n0 * cross, c1 = n1 * n1 * h + 2.0f * n1 * cross;
    const bool up = c1 < c0;
    fast = fabsf(cross) <= cv.y * sg && fabsf(tt) < GREEDY_TMAX;
    return up ? make_float2(g1, n1) : make_float2(g0, n0);
}

typedef float floatx4 __attribute__((ext_vector_type(4)));

// One super-block of a greedy pass (columns s0 .. s0 + sw, sw <= GSB) for
// GQR rows, one launch per super-block.  Csb [rows, GSB] holds
// err @ H[:, j] for the super-block's columns as of its start.  Block b's
// cross terms are Csb plus the changes D of the super-block's earlier
// blocks, D [16 rows, 64 b] kept in LDS, times H[earlier, block]: on the
// matrix cores as (H^T D^T) in 16 x 16 tiles, tile t holding the block
// columns 4 u + t (u = 0..15), the columns lane p = t owns, so that each lane
// fetches H[j'][j0 + 4 u .. + 3] as one vector for the four tiles.
// Two waves: wave 0 runs the blocks' columns; meanwhile wave 1 stages the
// next block's H tile and sums the next block's corrections from all but
// the current block, then, once the current block's changes are in LDS,
// adds those (one accumulation in block order).
// FULL: every block whole and the pitch of H a multiple of 4.  PE: per-element
// scales sc[rows, cols] (each lane keeps its columns' scales with their err
// and codes), else per-row scales sc[rows].
template <bool FULL, bool PE>
__global__ __launch_bounds__(128) void greedy_sb_kernel(float* err, float* Qf, const float* sc, const float* H,
                                                        int64_t ldh, const float* hd, const float* Csb,
                                                        int64_t rows, int64_t cols, int64_t s0, int sw, float qmin,
                                                        float qmax) {
    __shared__ __align__(16) float Hl[2][GB][GQ][GSLOT];   // Hl[b & 1][j'][p][m] = H[j0 + j'][j0 + 4 m + p]
    __shared__ __align__(16) float4 colv[2][GB];           // {H_jj, H_jj or NaN (guard), 1 / H_jj, 0}
    __shared__ __align__(16) float Dl[GSB][GQR];           // Dl[j - s0][row]: the block's change of err
    __shared__ __align__(16) float Xs[GQR][GQ][GSLOT];     // corrections of the next block, Xs[row][p][m]
    __shared__ float Gs[GQR][PE ? 4 : 3][GB];              // guarded rerun: err, codes, cross terms (, scales)
    const int w = threadIdx.x >> 6, t = threadIdx.x & 63;
    const int nblk = (sw + GB - 1) / GB;
    auto width = [&](int b) { return FULL ? GB : (int)min((int64_t)GB, (int64_t)sw - (int64_t)b * GB); };

    // ---- wave 1: H tiles and corrections ----
    auto put_tile = [&](int b) {   // H[blk, blk] of block b and its diagonal, into buffer b & 1
        const int64_t jb = s0 + (int64_t)b * GB;
        const int nbb = width(b);
        float hv[GB];
#pragma unroll
        for (int a = 0; a < GB; ++a) hv[a] = (FULL || (a < nbb && t < nbb)) ? H[(jb + a) * ldh + jb + t] : 0.0f;
        const float h = (FULL || t < nbb) ? (hd ? hd[jb + t] : H[(jb + t) * ldh + jb + t]) : 1.0f;
#pragma unroll
        for (int a = 0; a < GB; ++a) Hl[b & 1][a][t & (GQ - 1)][t / GQ] = hv[a];
        const bool hok = h >= 0x1p-60f && h <= 0x1p30f;
        colv[b & 1][t] = make_float4(h, hok ? h : __builtin_nanf(""), 1.0f / h, 0.0f);
    };
    floatx4 acc[GQ];
    const int lr = t & 15, lk = t >> 4;
    // acc += D[:, 4 ks .. 4 ks + 3] H[s0 + 4 ks .., block b] for ks in [k_lo, k_hi) (multiples of 16)
    auto corrections = [&](int b, int k_lo, int k_hi) {
        const int64_t c = s0 + (int64_t)b * GB + 4 * lr;
        auto hload = [&](int ks) -> float4 {
            const float* src = H + (s0 + 4 * ks + lk) * ldh + c;
            if (FULL) return *reinterpret_cast<const float4*>(src);
            return make_float4(c < cols ? src[0] : 0.0f, c + 1 < cols ? src[1] : 0.0f, c + 2 < cols ? src[2] : 0.0f,
                               c + 3 < cols ? src[3] : 0.0f);
        };
        constexpr int PF = 8;
        auto group = [&](int k0, const float4 (&hv)[PF]) {
            float bv[PF];
#pragma unroll
            for (int i = 0; i < PF; ++i) bv[i] = Dl[4 * (k0 + i) + lk][lr];
#pragma unroll
            for (int i = 0; i < PF; ++i) {
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(hv[i].x, bv[i], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(hv[i].y, bv[i], acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(hv[i].z, bv[i], acc[2], 0, 0, 0);
                acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(hv[i].w, bv[i], acc[3], 0, 0, 0);
            }
        };
        auto fetch = [&](int k0, float4 (&hv)[PF]) {   // clamped: past the range, in-bounds filler
#pragma unroll
            for (int i = 0; i < PF; ++i) hv[i] = hload(min(k0 + i, k_hi - 1));
            __builtin_amdgcn_sched_barrier(0);
        };
        float4 ha[PF], hb[PF];
        fetch(k_lo, ha);
        for (int k0 = k_lo; k0 < k_hi; k0 += 2 * PF) {
            fetch(k0 + PF, hb);
            group(k0, ha);
            fetch(k0 + 2 * PF, ha);
            group(k0 + PF, hb);
        }
    };

    // ---- wave 0: the columns ----
    const int p = t & (GQ - 1), rr = t / GQ;
    const int64_t r = (int64_t)blockIdx.x * GQR + rr;
    const bool live = w == 0 && r < rows;
    const float s = (live && !PE) ? sc[r] : 1.0f;
    const float is = 1.0f / s;
    const float sg = greedy_guard(s);
    float er[GSLOT], e0[GSLOT], qr[GSLOT], cr[GSLOT], sr[PE ? GSLOT : 1];
    auto load_raw = [&](int b) {   // block b's err, codes and super-block cross terms
        const int64_t j0 = s0 + (int64_t)b * GB;
        const int nb = width(b);
#pragma unroll
        for (int m = 0; m < GSLOT; ++m) {
            const int col = GQ * m + p;
            const bool ok = live && (FULL || col < nb);
            er[m] = ok ? err[r * cols + j0 + col] : 0.0f;
            qr[m] = ok ? Qf[r * cols + j0 + col] : 0.0f;
            cr[m] = ok ? Csb[r * GSB + (j0 - s0) + col] : 0.0f;
            if constexpr (PE) sr[m] = ok ? sc[r * cols + j0 + col] : 1.0f;
        }
    };
    auto add_corr = [&](int b) {
        if (b > 0) {
#pragma unroll
            for (int m = 0; m < GSLOT; ++m) cr[m] = cr[m] + Xs[rr][p][m];
        }
    };

    if (w == 1) put_tile(0);
    else load_raw(0);
    lds_barrier();
    for (int b = 0; b < nblk; ++b) {
        if (w == 0) {
            const int64_t j0 = s0 + (int64_t)b * GB;
            const int nb = width(b);
            const int buf = b & 1;
            add_corr(b);
#pragma unroll
            for (int m = 0; m < GSLOT; ++m) e0[m] = er[m];
            // Column jl of the block (jl a compile-time constant: register
            // slots).  A lane outside the window's domain only sets `bad`,
            // so the common path has no branch; the wave's rows are then run
            // again below.  Columns past a partial block (and rows past the
            // matrix) run on zeros (err, code, cross terms and H; H_jj = 1):
            // they decide code 0 with no change, add nothing to the real
            // columns and are not stored.
            uint64_t bad = 0;   // lanes that left the window's domain
            float4 cvn, hc[GSLOT / 4], hn[GSLOT / 4];   // column data and H row share, one column ahead
            const float4* Hl4 = reinterpret_cast<const float4*>(&Hl[buf][0][p][0]);
            const float4* cvp = &colv[buf][0];
            auto column = [&](auto JL) {
                constexpr int jl = decltype(JL)::value, m = jl / GQ, o = jl % GQ;
                const float4 cv = cvn;
                if constexpr (jl + 1 < GB) {
                    cvn = cvp[jl + 1];
#pragma unroll
                    for (int g = (jl + 1) / 16; g < GSLOT / 4; ++g) hn[g] = Hl4[(jl + 1) * (GQ * GSLOT / 4) + g];
                }
                const float xe = er[m];
                bool fast;
                float2 dec;
                if constexpr (PE) {
                    const float se = sr[m];
                    dec = greedy_decide(xe, qr[m], cr[m], cv, se, 1.0f / se, greedy_guard(se), qmin, qmax, fast);
                } else {
                    dec = greedy_decide(xe, qr[m], cr[m], cv, s, is, sg, qmin, qmax, fast);
                }
                bad |= __builtin_amdgcn_ballot_w64(!fast);
                __asm__ volatile("" : "+s"(bad));   // fold this column's test in now, not at the end
                const float d = quad_bcast<o>(dec.y - xe);
                if (p == o) {
                    er[m] = dec.y;
                    qr[m] = dec.x;
                }
                __asm__ volatile("" : "+v"(er[m]), "+v"(qr[m]));   // select now: keeps the columns' results dead
#pragma unroll
                for (int m2 = m; m2 < GSLOT; ++m2) {
                    const float4 h4 = hc[m2 / 4];
                    const float hv = m2 % 4 == 0 ? h4.x : m2 % 4 == 1 ? h4.y : m2 % 4 == 2 ? h4.z : h4.w;
                    cr[m2] = fmaf(d, hv, cr[m2]);
                }
#pragma unroll
                for (int g = 0; g < GSLOT / 4; ++g) hc[g] = hn[g];
                __builtin_amdgcn_sched_barrier(0);   // keep the one-column-ahead loads where they are
            };
            cvn = cvp[0];
#pragma unroll
            for (int g = 0; g < GSLOT / 4; ++g) hc[g] = Hl4[g];
            static_for<0, GB>(column);
            if (bad) {
                // Rare: the block again from its start for this wave's rows,
                // one lane per row, the same arithmetic in the same order,
                // with the whole-grid scan where the window does not apply.
                __asm__ volatile("" ::: "memory");   // reload, rather than keep the first loads live
                load_raw(b);
                add_corr(b);
#pragma unroll
                for (int m = 0; m < GSLOT; ++m) {
                    Gs[rr][0][GQ * m + p] = er[m];
                    Gs[rr][1][GQ * m + p] = qr[m];
                    Gs[rr][2][GQ * m + p] = cr[m];
                    if constexpr (PE) Gs[rr][PE ? 3 : 0][GQ * m + p] = sr[m];
                }
                lds_wave_fence();
                if (p == 0) {
                    for (int jl = 0; jl < nb; ++jl) {
                        const float4 cv = colv[buf][jl];
                        const float xe = Gs[rr][0][jl], xq = Gs[rr][1][jl];
                        const float se = PE ? Gs[rr][PE ? 3 : 0][jl] : s;
                        const float ise = PE ? 1.0f / se : is, sge = PE ? greedy_guard(se) : sg;
                        bool fast;
                        float2 dec = greedy_decide(xe, xq, Gs[rr][2][jl], cv, se, ise, sge, qmin, qmax, fast);
                        if (!fast) dec = greedy_scan(xe, xq, se, cv.x, Gs[rr][2][jl] - xe * cv.x, qmin, qmax);
                        Gs[rr][0][jl] = dec.y;
                        Gs[rr][1][jl] = dec.x;
                        const float d = dec.y - xe;
                        for (int j = jl + 1; j < nb; ++j)
                            Gs[rr][2][j] = fmaf(d, Hl[buf][jl][j % GQ][j / GQ], Gs[rr][2][j]);
                    }
                }
                lds_wave_fence();
#pragma unroll
                for (int m = 0; m < GSLOT; ++m) {
                    er[m] = Gs[rr][0][GQ * m + p];
                    qr[m] = Gs[rr][1][GQ * m + p];
                }
            }
#pragma unroll
            for (int m = 0; m < GSLOT; ++m) {
                const int col = GQ * m + p;
                if (b + 1 < nblk) Dl[b * GB + col][rr] = er[m] - e0[m];
                if (live && (FULL || col < nb)) {
                    err[r * cols + j0 + col] = er[m];
                    Qf[r * cols + j0 + col] = qr[m];
                }
            }
            if (b + 1 < nblk) load_raw(b + 1);   // in flight through the corrections
        } else if (b + 1 < nblk) {
#pragma unroll
            for (int u = 0; u < GQ; ++u) acc[u] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
            put_tile(b + 1);
            if (b > 0) corrections(b + 1, 0, 16 * b);
        }
        lds_barrier();   // block b's changes are in Dl, block b + 1's tile in place
        if (w == 1 && b + 1 < nblk) {
            corrections(b + 1, 16 * b, 16 * b + 16);
            // acc[u][v] = correction of row lr, column 4 (4 lk + v) + u
#pragma unroll
            for (int u = 0; u < GQ; ++u)
                *reinterpret_cast<float4*>(&Xs[lr][u][4 * lk]) = make_float4(acc[u][0], acc[u][1], acc[u][2], acc[u][3]);
        }
        lds_barrier();   // block b + 1's corrections are in Xs
    }
}

__global__ void to_int8_kernel(const float* Qf, int64_t n, float qmin, float qmax, int8_t* Q) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        Q[i] = (int8_t)(int)clampf(Qf[i], qmin, qmax);
}

static int egrid(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(cdiv(n, 256), 65536)); }

// hd[j] = H[j][j]
__global__ void diag_kernel(const float* H, int64_t n, float* hd) {
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x)
        hd[j] = H[j * n + j];
}

// US[i][c] = U[i][c] * s[c]   (n x k, U pitch ldu)
__global__ void scale_cols_kernel(const float* U, int64_t ldu, const float* s, int64_t n, int64_t k, float* US) {
    const int64_t total = n * k;
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = idx / k, c = idx - i * k;
        US[idx] = U[i * ldu + c] * s[c];
    }
}

// part[b] = sum over the block's share of err * EH (fp64), EH = err @ H
__global__ void proxy_partial_kernel(const float* err, const float* EH, int64_t n, double* part) {
    __shared__ double red[4];
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        acc += (double)err[i] * (double)EH[i];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

constexpr int PROXY_PARTS = 1024;

// Two-level pass.  Columns go in super-blocks of GSB: one GEMM gives the
// cross terms of a whole super-block, C = err @ Hc[sb, :]^T (K = cols, full
// tiles), and one launch of greedy_sb_kernel runs the super-block's 64-column
// blocks, adding each block's changes to the later blocks' cross terms on
// the way.  Cross terms of later super-blocks come from the updated err.
// Same sums as the reference's GEMM per block over all of err, in another
// fp32 order.
// The cross-term GEMM of a super-block has few 128-tiles (rows / 128 x 4)
// and a long K (= cols): it runs as GSPLIT products over K / GSPLIT each
// (GSPLIT times the tiles, two per CU), summed in order by split_sum_kernel.
constexpr int GSPLIT = 4;

// C[r][c] = ((P_0 + P_1) + P_2) + P_3 for the GSPLIT partial products
// (pitch GSB, stride rows * GSB).
__global__ void split_sum_kernel(const float* __restrict__ P, int64_t rows, int64_t sw, float* __restrict__ C) {
    const int64_t total = rows * sw, stride = rows * GSB;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / sw, c = i - r * sw, o = r * GSB + c;
        float v = P[o];
#pragma unroll
        for (int k = 1; k < GSPLIT; ++k) v = v + P[k * stride + o];
        C[o] = v;
    }
}

// The same sums of products of split operands, where an infinity gives a NaN:
// a 64 x 64 tile (a work-group) with a sum that is not finite is formed again
// as the fp32 product g, in place of P_0, and such sums are taken from there,
// so that a NaN in C is one of theirs.  (One infinity in every row, [2050,
// 2048], one pass: 7.3 ms, 35.7 with one thread summing the K products of such
// an element; 4.3 without infinities.  [4096, 4096]: 15.8 and 8.2 ms.)
__global__ __launch_bounds__(256) void split_sum_checked_kernel(const float* P, int64_t rows, int64_t sw, float* C,
                                                               GemmArgs g) {
    __shared__ __attribute__((aligned(16))) float lds[2 * gk::Geo<64>::TILE_F];
    const int64_t stride = rows * GSB, r0 = (int64_t)blockIdx.y * 64, c = (int64_t)blockIdx.x * 64 + (threadIdx.x & 63);
    auto finite = [](float v) { return fabsf(v) <= 3.402823466e38f; };
    bool bad = false;
#pragma unroll 4
    for (int u = 0; u < 16; ++u) {
        const int64_t r = r0 + 4 * u + (threadIdx.x >> 6), o = r * GSB + c;
        if (r >= rows || c >= sw) continue;
        float v = P[o];
#pragma unroll
        for (int k = 1; k < GSPLIT; ++k) v = v + P[k * stride + o];
        C[o] = v;
        bad |= !finite(v);
    }
    if (!__syncthreads_or(bad)) return;   // (every thread has read its part of P_0)
    gk::gemm_tile<0, 1, true, 64, gk::CHUNK_SUM>(g, gk::tile_range<64>(g, blockIdx.y, blockIdx.x), 0, lds);
    __syncthreads();
    for (int u = 0; u < 16; ++u) {
        const int64_t r = r0 + 4 * u + (threadIdx.x >> 6), o = r * GSB + c;
        if (r < rows && c < sw && !finite(C[o])) C[o] = P[o];
    }
}

// Large searches form the cross terms from split operands (split.hpp): H's
// planes once, err's kept up to date super-block by super-block.  The product
// of a super-block, bounded by the fp32 MFMA rate before, took 148 us at
// [4096, 4096] and takes 83 on the bf16 pipes, for 10 us of splitting.  The
// line, five passes (general -> split, us): [4096, 4096] 16900 -> 15209,
// [2048, 4096] 14026 -> 12851, [4096, 8192] 41900 -> 33934, [2048, 2048] 3662 ->
// 3511; but [1024, 4096] 11805 -> 11970, [64, 8192] 19108 -> 21390, where H's
// planes and a few tiles' latency cost more than the product.
constexpr int64_t GREEDY_SPLIT_COLS = 2048, GREEDY_SPLIT_ROWS = 2048, GREEDY_SPLIT_MAX_BYTES = 64LL << 30;
struct GreedyPlanes {
    SplitPlanes E, H;   // err by rows, H by rows
};
// Bytes of the planes (0: the general path), and (w) their places from `base` on.
static int64_t greedy_plane_bytes(int64_t rows, int64_t cols, char* base, GreedyPlanes* w) {
    if (cols % (GSPLIT * SP_ROWS) || cols < GREEDY_SPLIT_COLS || rows < GREEDY_SPLIT_ROWS) return 0;
    const int64_t kc = cols / SP_K, e = cdiv(rows, SP_ROWS) * kc * SP_CHUNK, h = cols / SP_ROWS * kc * SP_CHUNK;
    if ((e + h) * (int64_t)sizeof(uint16_t) > GREEDY_SPLIT_MAX_BYTES) return 0;
    if (w) {
        uint16_t* p = reinterpret_cast<uint16_t*>((reinterpret_cast<uintptr_t>(base) + 255) & ~(uintptr_t)255);
        w->E = SplitPlanes{p, SP_RECT, kc, 0};
        w->H = SplitPlanes{p + e, SP_RECT, kc, 0};
    }
    return (e + h) * (int64_t)sizeof(uint16_t) + 256;
}

// part: scratch for the split products (GSPLIT * rows * GSB floats), or null.
// sc / pe: the scales, per row (pe 0) or per element (pe 1).  pl: planes of err
// and Hc, or null.
static int greedy_pass(float* err, float* Qf, const float* sc, int pe, const float* Hc, const float* hd, float* C,
                       float* part, int64_t rows, int64_t cols, float qmin, float qmax, const GreedyPlanes* pl,
                       hipStream_t st) {
    for (int64_t s0 = 0; s0 < cols; s0 += GSB) {
        const int64_t sw = std::min<int64_t>(GSB, cols - s0);
        const int64_t ks = cols / GSPLIT;
        const bool split = part && cols % (GSPLIT * 128) == 0 && cdiv(rows, 128) * cdiv(sw, 128) < 256 &&
                           ks >= 1024;
        int rc;
        if (pl) {
            SplitGemm g{};
            g.M = rows;
            g.N = sw;
            g.K = ks;
            g.alpha = 1.0f;
            g.A.s = pl->E;
            g.B.s = pl->H;
            g.B.r0 = s0 / SP_ROWS;
            g.A.zc = g.B.zc = ks / SP_K;
            g.C = part;
            g.ldc = GSB;
            g.sC = rows * GSB;
            g.cmask = CMASK_FULL;
            g.krange = KR_FULL;
            g.batch = GSPLIT;
            g.tag = PT_SPLIT_GREEDY;
            g.algo_flops = 2.0 * rows * sw * cols;
            if ((rc = split_gemm(g, st))) return rc;
            const GemmArgs f{rows, sw, cols, 1.0f, 0.0f, err, cols, 0, Hc + s0 * cols, cols, 0, part, GSB, 0, 0, 1,
                             CMASK_FULL, KR_FULL, 1, PT_GEMM_GREEDY};
            hipLaunchKernelGGL(split_sum_checked_kernel, dim3((unsigned)cdiv(sw, 64), (unsigned)cdiv(rows, 64)),
                               dim3(256), 0, st, part, rows, sw, C, f);
            IC_CHECK_LAUNCH();
        } else if (split) {
            GemmArgs g{rows, sw, ks, 1.0f, 0.0f, err, cols, ks, Hc + s0 * cols, cols, ks, part, GSB, rows * GSB,
                       0, 1, CMASK_FULL, KR_FULL, GSPLIT, PT_GEMM_GREEDY};
            g.algo_flops = 2.0 * rows * sw * cols;
            if ((rc = gemm_f32(g, st))) return rc;
            hipLaunchKernelGGL(split_sum_kernel, dim3(egrid(rows * sw)), dim3(256), 0, st, part, rows, sw, C);
            IC_CHECK_LAUNCH();
        } else {
            GemmArgs g{rows, sw, cols, 1.0f, 0.0f, err, cols, 0, Hc + s0 * cols, cols, 0, C, GSB, 0, 0, 1,
                       CMASK_FULL, KR_FULL, 1, PT_GEMM_GREEDY};
            if ((rc = gemm_f32(g, st))) return rc;
        }
        {
            ProfScope prof_scope(st, PT_GREEDY, (double)rows * sw * (GB + 2.0 * sw), (double)rows * sw * 20);
            const bool full = sw % GB == 0 && cols % 4 == 0;
#define ICQ_GSB(F, P) hipLaunchKernelGGL((greedy_sb_kernel<F, P>), dim3((unsigned)cdiv(rows, GQR)), dim3(128), 0, st, \
                                         err, Qf, sc, Hc, cols, hd, C, rows, cols, s0, (int)sw, qmin, qmax)
            if (full) {
                if (pe) ICQ_GSB(true, true); else ICQ_GSB(true, false);
            } else {
                if (pe) ICQ_GSB(false, true); else ICQ_GSB(false, false);
            }
#undef ICQ_GSB
            IC_CHECK_LAUNCH();
        }
        if (pl) {   // the columns that changed
            int rc2 = split_planes(err, rows, cols, 0, 0, rows, s0, s0 + sw, 0, 0, pl->E, 1, st, 1, 0,
                                   cols);
            if (rc2) return rc2;
        }
    }
    return IC_OK;
}

}  // namespace icq

using namespace icq;

extern "C" int ic_ldlq_init_scales(const float* row_absmax, int64_t rows, int64_t cols, int bits, float* srow,
                                   float* S, void* stream) {
    IC_REQUIRE(row_absmax && S, "ic_ldlq_init_scales: null pointer");
    if (rows * cols == 0) return IC_OK;
    hipLaunchKernelGGL(ldlq_init_scales_kernel, dim3(egrid(rows * cols)), dim3(256), 0, as_stream(stream),
                       row_absmax, rows, cols, bits == 8 ? 127.0f : 7.0f, srow, S);
    IC_CHECK_LAUNCH();
    return IC_OK;
}

extern "C" int ic_sanitize_scales(float* S, int64_t n, void* stream) {
    IC_REQUIRE(S, "ic_sanitize_scales: null pointer");
    if (n == 0) return IC_OK;
    hipLaunchKernelGGL(sanitize_scales_kernel, dim3(egrid(n)), dim3(256), 0, as_stream(stream), S, n);
    IC_CHECK_LAUNCH();
    return IC_OK;
}

extern "C" int ic_ldlq_mse(const float* W, const int8_t* Q, const float* S, int64_t n, double* out_sumsq,
                           void* workspace, void* stream) {
    IC_REQUIRE(W && Q && S && out_sumsq && workspace, "ic_ldlq_mse: null pointer");
    hipStream_t st = as_stream(stream);
    double* part = reinterpret_cast<double*>(workspace);
    hipLaunchKernelGGL(ldlq_mse_kernel, dim3(1024), dim3(256), 0, st, W, Q, S, n, part);
    IC_CHECK_LAUNCH();
    hipLaunchKernelGGL(sum_parts_kernel, dim3(1), dim3(256), 0, st, part, 1024, out_sumsq);
    IC_CHECK_LAUNCH();
    return IC_OK;
}

extern "C" int ic_ldlq_update_scales(const float* W, const int8_t* Q, const float* cur, const float* flat, int64_t n,
                                     float momentum, float lo, float hi, float* out, void* stream) {
    IC_REQUIRE(W && Q && cur && flat && out, "ic_ldlq_update_scales: null pointer");
    if (n == 0) return IC_OK;
    hipLaunchKernelGGL(ldlq_update_kernel, dim3(egrid(n)), dim3(256), 0, as_stream(stream), W, Q, cur, flat, n,
                       momentum, lo, hi, out);
    IC_CHECK_LAUNCH();
    return IC_OK;
}

extern "C" int ic_ls_scales(const int8_t* Q, const float* W, int64_t rows, int64_t cols, float* out, void* stream) {
    IC_REQUIRE(Q && W && out && rows < (1LL << 31), "ic_ls_scales: bad arguments");
    if (rows == 0) return IC_OK;
    hipLaunchKernelGGL(ls_scales_kernel, dim3((unsigned)cdiv(rows, 4)), dim3(256), 0, as_stream(stream), Q, W, rows,
                       cols, out);
    IC_CHECK_LAUNCH();
    return IC_OK;
}

extern "C" int64_t ic_greedy_min_workspace_bytes(int64_t rows, int64_t cols) {
    return (2 * rows * cols + rows * GSB + GSPLIT * rows * GSB) * (int64_t)sizeof(float) + 256;
}

extern "C" int64_t ic_greedy_workspace_bytes(int64_t rows, int64_t cols) {
    return ic_greedy_min_workspace_bytes(rows, cols) + greedy_plane_bytes(rows, cols, nullptr, nullptr);
}

extern "C" int ic_greedy_sized(const float* W, int8_t* Q, const float* scale, int scale_kind, const float* H,
                               int64_t rows, int64_t cols, int passes, int bits, void* workspace,
                               int64_t workspace_bytes, void* stream) {
    IC_REQUIRE(W && Q && scale && H && workspace, "ic_greedy: null pointer");
    IC_REQUIRE(bits == 4 || bits == 8, "ic_greedy: bits must be 4 or 8");
    IC_REQUIRE(scale_kind == 0 || scale_kind == 1, "ic_greedy: scale_kind must be 0 (per row) or 1 (per element)");
    if (rows == 0 || cols == 0 || passes <= 0) return IC_OK;
    IC_REQUIRE(workspace_bytes >= ic_greedy_min_workspace_bytes(rows, cols), "ic_greedy: workspace too small");
    hipStream_t st = as_stream(stream);
    const float qmin = bits == 4 ? -8.0f : -128.0f, qmax = bits == 4 ? 7.0f : 127.0f;
    float* err = reinterpret_cast<float*>(workspace);
    float* Qf = err + rows * cols;
    float* cross = Qf + rows * cols;
    hipLaunchKernelGGL(greedy_err_kernel, dim3(egrid(rows * cols)), dim3(256), 0, st, Q, scale, scale_kind, W, rows,
                       cols, err, Qf);
    IC_CHECK_LAUNCH();
    float* part = cross + rows * GSB;
    GreedyPlanes planes, *pl = nullptr;
    if (workspace_bytes >= ic_greedy_workspace_bytes(rows, cols) &&
        greedy_plane_bytes(rows, cols, reinterpret_cast<char*>(part + GSPLIT * rows * GSB), &planes)) {
        pl = &planes;
        int rc = split_planes(H, cols, cols, 0, 0, cols, 0, cols, 0, 0, pl->H, 1, st);
        if (!rc)
            rc = split_planes(err, rows, cols, 0, 0, rows, 0, cols, 0, 0, pl->E, 1, st, 1, 0, cols);
        if (rc) return rc;
    }
    for (int p = 0; p < passes; ++p) {
        int rc = greedy_pass(err, Qf, scale, scale_kind, H, nullptr, cross, part, rows, cols, qmin, qmax, pl, st);
        if (rc) return rc;
    }
    hipLaunchKernelGGL(to_int8_kernel, dim3(egrid(rows * cols)), dim3(256), 0, st, Qf, rows * cols, qmin, qmax, Q);
    IC_CHECK_LAUNCH();
    return IC_OK;
}

extern "C" int ic_greedy(const float* W, int8_t* Q, const float* scale, int scale_kind, const float* H, int64_t rows,
                         int64_t cols, int passes, int bits, void* workspace, void* stream) {
    return ic_greedy_sized(W, Q, scale, scale_kind, H, rows, cols, passes, bits, workspace,
                           ic_greedy_workspace_bytes(rows, cols), stream);
}

extern "C" int64_t ic_greedy_lowrank_workspace_bytes(int64_t rows, int64_t cols, int64_t k) {
    return (3 * rows * cols + rows * GSB + cols * cols + cols * std::max<int64_t>(k, 1) + cols +
            GSPLIT * rows * GSB) * (int64_t)sizeof(float) + PROXY_PARTS * (int64_t)sizeof(double) + 1024;
}

extern "C" int ic_greedy_lowrank(const float* W, int8_t* Q, const float* scale, int scale_kind, const float* H,
                                 const float* U, int64_t ldu, const float* s, int64_t k, int64_t rows, int64_t cols,
                                 int passes, int bits, int* passes_run, void* workspace, void* stream) {
    IC_REQUIRE(W && Q && scale && H && workspace && (k == 0 || (U && s)), "ic_greedy_lowrank: null pointer");
    IC_REQUIRE(bits == 4 || bits == 8, "ic_greedy_lowrank: bits must be 4 or 8");
    IC_REQUIRE(scale_kind == 0 || scale_kind == 1,
               "ic_greedy_lowrank: scale_kind must be 0 (per row) or 1 (per element)");
    IC_REQUIRE(k >= 0 && k <= cols && ldu >= k, "ic_greedy_lowrank: bad rank");
    if (passes_run) *passes_run = 0;
    if (rows == 0 || cols == 0 || passes <= 0) return IC_OK;
    hipStream_t st = as_stream(stream);
    const float qmin = bits == 4 ? -8.0f : -128.0f, qmax = bits == 4 ? 7.0f : 127.0f;
    float* err = reinterpret_cast<float*>(workspace);
    float* Qf = err + rows * cols;
    float* EH = Qf + rows * cols;
    float* cross = EH + rows * cols;
    float* Hk = cross + rows * GSB;
    float* US = Hk + cols * cols;
    float* hd = US + cols * std::max<int64_t>(k, 1);
    float* split_part = hd + cols;
    double* part = reinterpret_cast<double*>(
        (reinterpret_cast<uintptr_t>(split_part + GSPLIT * rows * GSB) + 255) & ~(uintptr_t)255);
    // Hk = U_k diag(s_k) U_k^T
    if (k == 0) {
        IC_CHECK_HIP(hipMemsetAsync(Hk, 0, cols * cols * sizeof(float), st));
    } else {
        hipLaunchKernelGGL(scale_cols_kernel, dim3(egrid(cols * k)), dim3(256), 0, st, U, ldu, s, cols, k, US);
        IC_CHECK_LAUNCH();
        GemmArgs g{cols, cols, k, 1.0f, 0.0f, US, k, 0, U, ldu, 0, Hk, cols, 0, 0, 1, CMASK_FULL, KR_FULL, 1,
                   PT_GEMM_GREEDY};
        int rc = gemm_f32(g, st);
        if (rc) return rc;
    }
    hipLaunchKernelGGL(diag_kernel, dim3(egrid(cols)), dim3(256), 0, st, H, cols, hd);
    IC_CHECK_LAUNCH();
    hipLaunchKernelGGL(greedy_err_kernel, dim3(egrid(rows * cols)), dim3(256), 0, st, Q, scale, scale_kind, W, rows,
                       cols, err, Qf);
    IC_CHECK_LAUNCH();
    double prev = 0.0;
    int done = 0;
    for (int p = 0; p < passes; ++p) {
        int rc = greedy_pass(err, Qf, scale, scale_kind, Hk, hd, cross, split_part, rows, cols, qmin, qmax, nullptr,
                             st);
        if (rc) return rc;
        done = p + 1;
        if (p + 1 == passes) break;   // a stall test after the last pass changes nothing
        // proxy = sum((err @ H) * err) with the full Hessian
        GemmArgs g{rows, cols, cols, 1.0f, 0.0f, err, cols, 0, H, cols, 0, EH, cols, 0, 0, 0, CMASK_FULL, KR_FULL,
                   1, PT_GEMM_GREEDY};
        if ((rc = gemm_f32(g, st))) return rc;
        hipLaunchKernelGGL(proxy_partial_kernel, dim3(PROXY_PARTS), dim3(256), 0, st, err, EH, rows * cols, part);
        IC_CHECK_LAUNCH();
        double parts[PROXY_PARTS];
        IC_CHECK_HIP(hipMemcpyAsync(parts, part, sizeof(parts), hipMemcpyDeviceToHost, st));
        IC_CHECK_HIP(hipStreamSynchronize(st));
        double proxy = 0.0;
        for (int i = 0; i < PROXY_PARTS; ++i) proxy += parts[i];
        if (p > 0 && proxy >= prev * 0.99) break;   // STALL_THRESHOLD (converter/config.py:128)
        prev = proxy;
    }
    if (passes_run) *passes_run = done;
    hipLaunchKernelGGL(to_int8_kernel, dim3(egrid(rows * cols)), dim3(256), 0, st, Qf, rows * cols, qmin, qmax, Q);
    IC_CHECK_LAUNCH();
    return IC_OK;
}

// Products of fp32 matrices as six bf16 MFMA products of split operands, and
// the kernels that split them (layout and terms: split.hpp).
//
// Bound by the matrix cores' power: a loop of v_mfma_f32_32x32x16_bf16 on
// registers reaches 2.48 PFLOP/s on zeros and 1.94 on uniform random operands
// (a sixth of which is the fp32 rate), and the 12288 inverse keeps the matrix
// cores 71 % busy in its merges and X^T X, 55 % in its K = 1024 updates, at
// the clock that leaves.  Against v_mfma_f32_16x16x4_f32 (gemm_dev.hpp) on the
// 12288 x 12288 inverse: X^T X 4.99 -> 3.58 ms (173 TFLOP/s of fp32 work),
// K = 1024 update of 11264 rows 1.14 -> 0.67 ms (196), merge T = L21 X11 of
// 4096 x 8192 1.69 -> 1.30 ms (211); the inverse 20.9 -> 16.1 ms.  Its error
// against 64 bits is lower (relative 2.98e-7, was 3.27e-7): an accumulator is
// rounded six times per 16 k, not once per k.
//
// split_gemm_kernel: work-group of 4 waves, 128 x 128 tile, each wave 64 x 64
// as 2 x 2 accumulators.  A stage is one chunk of each operand (16 k, 2 x 12
// KB, contiguous): 24 MFMAs of 32 cycles per wave against 12 16-byte LDS
// reads.  Stages are copied to LDS without passing through registers, into
// three buffers; a wave reads the next stage's operands behind the current
// one's MFMAs (reading them in the same stage: 703 us where this takes 670;
// through registers: 734).  Two work-groups per CU.  Every 128 k the
// accumulators are folded into a running sum (as in gemm_dev.hpp), which
// bounds the rounding error of long sums.  Running triangles in square
// blocks of tiles per XCD measured the same (the operands' rereads are not
// what limits it).
//
// MFMA 32x32x16 bf16 operand layout (lane l of 64):
//   A: A[i = l%32][k = 8 (l/32) + e]    B: B[k = 8 (l/32) + e][j = l%32]
//   D (16 values v): D[i = 8 (v/4) + 4 (l/32) + v%4][j = l%32]
#include "gemm_dev.hpp"
#include "split.hpp"

namespace icq {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef uint32_t uintx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void split3(float x, __bf16& a, __bf16& b, __bf16& c) {
    a = (__bf16)x;
    const float r = x - (float)a;    // exact
    b = (__bf16)r;
    c = (__bf16)(r - (float)b);      // exact
}

__device__ __forceinline__ uint16_t* op_ptr(const SplitOp& o, int64_t z, int64_t r, int64_t c) {
    return o.s.p + z * o.zp + split_chunk(o.s, o.r0 + z * o.zr + r, o.c0 + z * o.zc + c) * SP_CHUNK;
}

constexpr int SP_VEC = SP_CHUNK / 8;         // 16-byte vectors of a chunk: 768
constexpr int SP_BUFS = 3;                    // LDS buffers: one in registers or read, two under way
constexpr int SP_STAGE = 2 * SP_VEC;         // vectors of a stage
constexpr int SP_FOLD = 128 / SP_K;          // stages per accumulation chunk

// 16 bytes per lane from `src` to LDS, the wave's 1 KB at byte address `dst`
// (uniform), without passing through registers.  Waited for with vmcnt.
__device__ __forceinline__ void copy_to_lds(uint32_t dst, const uintx4* src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src) : "memory", "m0");
}

// At most N of the wave's copies (and other memory operations) outstanding.
template <int N>
__device__ __forceinline__ void wait_copies() {
    static_assert(N < 64, "vmcnt");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <bool SUB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void split_gemm_kernel(SplitGemm g,
                                                                                               GemmArgs geo,
                                                                                               int64_t ntiles,
                                                                                               int xcd) {
    __shared__ uintx4 lds[SP_BUFS * SP_STAGE];
    gk::TileRange tr;
    const int64_t z = blockIdx.z;
    if (xcd) {
        if (!gk::xcd_tile<128>(geo, blockIdx.x, tr)) return;
    } else {
        if ((int64_t)blockIdx.x >= ntiles) return;
        tr = gk::tile_of<128>(geo, blockIdx.x);
    }
    if (tr.skip) return;
    const int64_t ti = tr.i0 / SP_ROWS, tj = tr.j0 / SP_ROWS;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wi = (wave >> 1) * 64, wj = (wave & 1) * 64;   // uniform in the wave
    const int li = lane & 31, lo = lane >> 5;
    const int nst = (int)((tr.khi - tr.klo) / SP_K);
    const uintx4* pa = reinterpret_cast<const uintx4*>(op_ptr(g.A, z, ti, tr.klo / SP_K)) + t;
    const uintx4* pb = reinterpret_cast<const uintx4*>(op_ptr(g.B, z, tj, tr.klo / SP_K)) + t;
    float* C = g.C ? g.C + z * g.sC : nullptr;
    // element v of accumulator (a, b) is C[i0 + wi + 32 a + 8 (v/4) + v%4 + 4 lo][j0 + wj + 32 b + li]: a uniform
    // address and one offset per lane
    const uint32_t coff = 4 * lo * (uint32_t)g.ldc + li;
    auto crow = [&](float* base, int a, int b, int v) -> float* {
        return base + (tr.i0 + wi + 32 * a + 8 * (v >> 2) + (v & 3)) * g.ldc + (tr.j0 + wj + 32 * b);
    };
    const bool inside = tr.i0 + 128 <= g.M && tr.j0 + 128 <= g.N && (g.cmask == CMASK_FULL || ti != tj);
    auto stored = [&](int a, int b, int v) -> bool {
        const int64_t i = tr.i0 + wi + 32 * a + 8 * (v >> 2) + 4 * lo + (v & 3), j = tr.j0 + wj + 32 * b + li;
        return i < g.M && j < g.N && !(g.cmask == CMASK_LOWER && i < j) && !(g.cmask == CMASK_UPPER && i > j);
    };

    floatx16 acc[2][2], run[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = run[a][b][v] = 0.0f;
    if (SUB) {
        // the running result starts as C
        if (inside) {
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int v = 0; v < 16; ++v) run[a][b][v] = crow(C, a, b, v)[coff];
        } else {
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        if (stored(a, b, v)) run[a][b][v] = crow(C, a, b, v)[coff];
        }
    }
    // byte address in LDS of this wave's first 1 KB of buffer 0; a stage is 3 KB of each operand per wave
    const uint32_t lbase = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)(void*)&lds[0] + wave * 1024;
    auto stage_in = [&](int buf) {
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            copy_to_lds(lbase + buf * SP_STAGE * 16 + p * 4096, pa + p * 256);
            copy_to_lds(lbase + buf * SP_STAGE * 16 + SP_VEC * 16 + p * 4096, pb + p * 256);
        }
        pa += SP_VEC;
        pb += SP_VEC;
    };
    const uintx4* As = &lds[lo * 128 + wi + li];
    const uintx4* Bs = &lds[SP_VEC + lo * 128 + wj + li];
    struct Frags { bf16x8 a[3][2], b[3][2]; };
    auto read = [&](int buf, Frags& f) {
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                f.a[p][x] = __builtin_bit_cast(bf16x8, As[buf * SP_STAGE + p * 256 + 32 * x]);
                f.b[p][x] = __builtin_bit_cast(bf16x8, Bs[buf * SP_STAGE + p * 256 + 32 * x]);
            }
    };
    if (nst > 0) {
        // stages 0 .. SP_BUFS - 1 under way; the first operands in registers
#pragma unroll
        for (int s = 0; s < SP_BUFS; ++s) stage_in(s);
        wait_copies<6 * (SP_BUFS - 1)>();
        lds_barrier();
        Frags f0, f1;
        read(0, f0);
        int buf = 0;   // buffer of stage s
        // Step s: stage s + 1 has arrived for every wave (the SP_BUFS - 2 after
        // it may still be under way), and every wave has stage s in
        // registers, so stage s + SP_BUFS may overwrite its buffer; stage s + 1
        // is read behind stage s's MFMAs.
        auto step = [&](int s, Frags& f, Frags& nx) {
            const int b1 = buf == SP_BUFS - 1 ? 0 : buf + 1;
            if (s + SP_BUFS - 1 < nst) wait_copies<6 * (SP_BUFS - 2)>();
            else wait_copies<0>();
            lds_barrier();
            if (s + SP_BUFS < nst) stage_in(buf);
            read(b1, nx);   // (past the last stage: old contents, not used)
            // small terms first
#define ICQ_TERM(PA, PB)                                                                                  \
    _Pragma("unroll") for (int a = 0; a < 2; ++a) _Pragma("unroll") for (int b = 0; b < 2; ++b) acc[a][b] = \
        __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[PA][a], f.b[PB][b], acc[a][b], 0, 0, 0)
            ICQ_TERM(2, 0);
            ICQ_TERM(0, 2);
            ICQ_TERM(1, 1);
            ICQ_TERM(1, 0);
            ICQ_TERM(0, 1);
            ICQ_TERM(0, 0);
#undef ICQ_TERM
            buf = b1;
        };
        for (int s = 0; s < nst; s += SP_FOLD) {
#pragma unroll
            for (int u = 0; u < SP_FOLD; u += 2) {
                step(s + u, f0, f1);
                step(s + u + 1, f1, f0);
            }
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        run[a][b][v] = SUB ? run[a][b][v] - acc[a][b][v] : run[a][b][v] + acc[a][b][v];
                        acc[a][b][v] = 0.0f;
                    }
        }
    }
    if (!SUB && g.alpha < 0.0f) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v) run[a][b][v] = -run[a][b][v];
    }
    if (C) {
        if (inside) {
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int v = 0; v < 16; ++v) crow(C, a, b, v)[coff] = run[a][b][v];
        } else {
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int v = 0; v < 16; ++v)
                        if (stored(a, b, v)) crow(C, a, b, v)[coff] = run[a][b][v];
        }
    }
    if (g.out.s.p) {
        // planes of the transpose: a lane's four consecutive rows of one
        // column are half an octet
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int k = wi + 32 * a + 8 * q;   // first of the octet's 8 rows of the tile
                    uint16_t* ch = op_ptr(g.out, z, tj, ti * SP_PER_BLOCK + k / SP_K);
                    bf16x4 w[3];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        __bf16 x0, x1, x2;
                        split3(run[a][b][4 * q + e], x0, x1, x2);
                        w[0][e] = x0;
                        w[1][e] = x1;
                        w[2][e] = x2;
                    }
                    const int at = ((k & 8) / 8 * SP_ROWS + wj + 32 * b + li) * 8 + 4 * lo;
#pragma unroll
                    for (int p = 0; p < 3; ++p) *reinterpret_cast<bf16x4*>(ch + p * (SP_CHUNK / 3) + at) = w[p];
                }
    }
}

// One 16-byte vector of each plane per thread and step: 8 consecutive k of
// one chunk row.  Work-group: one 128 x 128 block of A (8 chunks).
__device__ __forceinline__ void store_octet(uint16_t* chunk, int oct, int row, const float (&x)[8]) {
    bf16x8 w[3];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        __bf16 a, b, c;
        split3(x[e], a, b, c);
        w[0][e] = a;
        w[1][e] = b;
        w[2][e] = c;
    }
#pragma unroll
    for (int p = 0; p < 3; ++p)
        *reinterpret_cast<bf16x8*>(chunk + p * (SP_CHUNK / 3) + (oct * SP_ROWS + row) * 8) = w[p];
}

// grid (column blocks, row blocks, squares x batch): the blocks from
// (rb0, cb0), of `squares` such regions `step` blocks apart along the diagonal.
template <bool TRANS, bool VEC>
__global__ __launch_bounds__(256) void split_planes_kernel(const float* A, int64_t n, int64_t nc, int64_t ld,
                                                          int64_t sA, int64_t rb0, int64_t cb0, int lower, int squares,
                                                          int64_t step, SplitPlanes out) {
    const int64_t m = blockIdx.z / squares, sq = blockIdx.z - m * squares;
    const int64_t rb = rb0 + blockIdx.y + sq * step, cb = cb0 + blockIdx.x + sq * step;
    if ((lower && cb > rb) || rb * SP_ROWS >= n) return;
    const float* P = A + m * sA;
    uint16_t* o = out.p + m * out.stride +
                  (TRANS ? split_chunk(out, cb, rb * SP_PER_BLOCK) : split_chunk(out, rb, cb * SP_PER_BLOCK)) * SP_CHUNK;
    const int t = threadIdx.x;
#pragma unroll 2
    for (int u = 0; u < 8; ++u) {
        const int idx = t + 256 * u;   // 2048 vectors of 8 values
        float x[8];
        int row, oct;                  // chunk row, octet of k (0..15) in the block
        if (TRANS) {
            row = idx & 127;
            oct = idx >> 7;
            const int64_t j = cb * SP_ROWS + row;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int64_t i = rb * SP_ROWS + oct * 8 + e;
                x[e] = i < n && j < nc ? P[i * ld + j] : 0.0f;
            }
        } else {
            oct = (idx & 7) + 8 * (idx >> 10);
            row = (idx >> 3) & 127;
            const int64_t i = rb * SP_ROWS + row, j = cb * SP_ROWS + oct * 8;
            if (VEC && i < n && j + 8 <= nc) {
                const float4 a = *reinterpret_cast<const float4*>(&P[i * ld + j]);
                const float4 b = *reinterpret_cast<const float4*>(&P[i * ld + j + 4]);
                x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
                x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = i < n && j + e < nc ? P[i * ld + j + e] : 0.0f;
            }
        }
        store_octet(o + (oct >> 1) * SP_CHUNK, oct & 1, row, x);
    }
}

}  // namespace

int split_gemm(const SplitGemm& g, hipStream_t st) {
    if (g.M <= 0 || g.N <= 0 || g.batch <= 0) return IC_OK;
    IC_REQUIRE(g.K % SP_ROWS == 0 && (g.alpha == 1.0f || g.alpha == -1.0f), "split_gemm: bad K or alpha");
    IC_REQUIRE(!g.sub || (g.C && g.alpha == -1.0f), "split_gemm: subtraction needs C and alpha = -1");
    GemmArgs geo{};
    geo.M = g.M;
    geo.N = g.N;
    geo.K = g.K;
    geo.cmask = g.cmask;
    geo.krange = g.krange;
    bool tri;
    const int64_t tiles = gk::tile_count<128>(geo, tri);
    const int64_t tm = cdiv(g.M, 128), tn = cdiv(g.N, 128);
    const int xcd = (!tri && tm >= gk::NXCD) ? 1 : 0;
    const int64_t grid = xcd ? cdiv(tm, gk::NXCD) * tn * gk::NXCD : tiles;
    IC_REQUIRE(grid < (1LL << 23) && g.batch <= 65535, "split_gemm: problem too large");
    ProfScope prof_scope(st, g.tag, g.algo_flops, 6.0 * g.batch * (g.M + g.N) * g.K + 4.0 * g.batch * g.M * g.N);
    const dim3 gd((unsigned)grid, 1, (unsigned)g.batch);
    if (g.sub) hipLaunchKernelGGL((split_gemm_kernel<true>), gd, dim3(256), 0, st, g, geo, tiles, xcd);
    else hipLaunchKernelGGL((split_gemm_kernel<false>), gd, dim3(256), 0, st, g, geo, tiles, xcd);
    IC_CHECK_LAUNCH();
    return IC_OK;
}

int split_planes(const float* A, int64_t n, int64_t ld, int64_t sA, int64_t r0, int64_t r1, int64_t c0, int64_t c1,
                 int transpose, int lower, const SplitPlanes& out, int64_t batch, hipStream_t st, int64_t squares,
                 int64_t step, int64_t ncols) {
    if (r1 <= r0 || c1 <= c0 || batch <= 0) return IC_OK;
    IC_REQUIRE(r0 % SP_ROWS == 0 && c0 % SP_ROWS == 0, "split_planes: unaligned block");
    const int64_t rbs = cdiv(r1 - r0, SP_ROWS), cbs = cdiv(c1 - c0, SP_ROWS);
    IC_REQUIRE(step % SP_ROWS == 0 && rbs <= 65535 && batch * squares <= 65535, "split_planes: problem too large");
    const bool vec = ((uintptr_t)A % 16) == 0 && ld % 4 == 0 && sA % 4 == 0;
    ProfScope prof_scope(st, PT_SPLIT_PLANES, 0.0, 10.0 * batch * squares * (r1 - r0) * (c1 - c0));
    const dim3 gd((unsigned)cbs, (unsigned)rbs, (unsigned)(batch * squares));
    const int64_t rb0 = r0 / SP_ROWS, cb0 = c0 / SP_ROWS;
    if (ncols < 0) ncols = n;
#define ICQ_SPLIT(TR, VE)                                                                                   \
    hipLaunchKernelGGL((split_planes_kernel<TR, VE>), gd, dim3(256), 0, st, A, n, ncols, ld, sA, rb0, cb0, \
                       lower, (int)squares, step / SP_ROWS, out)
    if (transpose) ICQ_SPLIT(true, false);
    else if (vec) ICQ_SPLIT(false, true);
    else ICQ_SPLIT(false, false);
#undef ICQ_SPLIT
    IC_CHECK_LAUNCH();
    return IC_OK;
}

}  // namespace icq

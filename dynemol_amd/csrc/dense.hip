// Dense FP64 algebra for the orthogonalisation S = L L^T, L^-1 and
// H_orth = L^-1 h L^-T, on gfx950 matrix cores (v_mfma_f64_16x16x4f64).
//
// Replaces the reference's S^-1 (dsytrf/dsytri on the CPU, MAGMA
// dgetrf/dgetri on the GPU: GPU_Interface.cpp:880-949) and H' = S^-1 h
// (xPU_dsymm / cublasDsymm: GPU_Interface.cpp:574-627, Taylor_gpu.cpp:695).
// All matrices are column-major with a leading dimension padded to a multiple
// of 64; the padding of S carries an identity block, so every blocked
// routine runs on whole 64 x 64 tiles.
#include "common.hpp"
#include "gemm.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace dh {

// C = alpha * opA(A) opB(B) + beta * C on T x T tiles, T = 64 or 32
// (gemm_accumulate).  A pair of 128 x 128 tiles per workgroup, which this
// replaces, took 112 us where N = 576 now takes 14, 474 for L^-1 h at 2112 (175
// now) and 1416 at 4096 (1110 now).
//
// Workgroups start in blockIdx order (x fastest).  With a k range that grows
// with the row (column) tile, columns (rows) run fastest and the longest tiles
// start first, so that the last ones to start are short; consecutive
// workgroups go round the XCDs, so an XCD keeps to an eighth of the fast
// dimension where that divides by 8 and its tiles share operands in its L2.
template <int T, int GK, int TA, int TB>
__global__ __launch_bounds__(256) void gemm_f64_kernel(Gemm g) {
    __shared__ double As[2][GK * T];
    __shared__ double Bs[2][GK * T];
    constexpr int MB = T / 32;
    const bool rows_fast = g.kmode == K_BELOW_COLTILE || g.kmode == K_FROM_COLTILE || g.kmode == K_FULL;
    int bi = rows_fast ? blockIdx.x : blockIdx.y, bj = rows_fast ? blockIdx.y : blockIdx.x;
    if (g.kmode == K_BELOW_ROWTILE) bi = gridDim.y - 1 - bi;
    else if (g.kmode == K_BELOW_COLTILE) bj = gridDim.y - 1 - bj;
    const int i0 = bi * T, j0 = bj * T;
    if (g.lower_only && i0 / TILE < j0 / TILE) return;
    const double* A = g.A + (long)blockIdx.z * g.strideA + (TA ? g.lda * (long)i0 : (long)i0);
    const double* B = g.B + (long)blockIdx.z * g.strideB + (TB ? (long)j0 : g.ldb * (long)j0);
    double* C = g.C + (long)blockIdx.z * g.strideC;
    int klo = 0, khi = g.K;
    if (g.kmode == K_BELOW_ROWTILE) khi = min(g.K, i0 + T);
    else if (g.kmode == K_BELOW_COLTILE) khi = min(g.K, j0 + T);
    else if (g.kmode == K_FROM_ROWTILE) klo = i0;
    else if (g.kmode == K_FROM_COLTILE) klo = j0;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int ib = i0 + (w >> 1) * (T / 2) + (lane & 15), jb = j0 + (w & 1) * (T / 2) + (lane >> 4);
    v4d acc[MB][MB];
    // C <- C - A B: the accumulators start at -C, whose latency overlaps the
    // first operand loads, and their negative is stored (exact either way)
    const bool cacc = g.c_acc != 0;
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int gi = min(ib + a * 16, g.M - 1), gj = min(jb + b * 16 + 4 * v, g.N - 1);
                acc[a][b][v] = cacc ? -C[gi + g.ldc * (long)gj] : 0.0;
            }
    gemm_accumulate<T, GK, TA, TB, false>(acc, A, g.lda, g.M - i0, B, g.ldb, g.N - j0, klo, khi, As, Bs,
                                          [](int, int) { return true; }, [](int j) { return j; });
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int gi = ib + a * 16, gj = jb + b * 16 + 4 * v;
                if (gi < g.M && gj < g.N) {
                    const long idx = gi + g.ldc * (long)gj;
                    if (cacc) {
                        C[idx] = -acc[a][b][v];
                    } else {
                        const double old = g.beta == 0.0 ? 0.0 : g.beta * C[idx];
                        C[idx] = g.alpha * acc[a][b][v] + old;
                    }
                }
            }
}

template <int T, int GK>
static void gemm_tiles(const Gemm& g, hipStream_t st) {
    const unsigned nr = (g.M + T - 1) / T, nc = (g.N + T - 1) / T, nz = g.batch > 0 ? g.batch : 1;
    const bool rows_fast = g.kmode == K_BELOW_COLTILE || g.kmode == K_FROM_COLTILE || g.kmode == K_FULL;
    const dim3 grid(rows_fast ? nr : nc, rows_fast ? nc : nr, nz);
    if (!g.transA && !g.transB) hipLaunchKernelGGL((gemm_f64_kernel<T, GK, 0, 0>), grid, dim3(256), 0, st, g);
    else if (!g.transA) hipLaunchKernelGGL((gemm_f64_kernel<T, GK, 0, 1>), grid, dim3(256), 0, st, g);
    else if (!g.transB) hipLaunchKernelGGL((gemm_f64_kernel<T, GK, 1, 0>), grid, dim3(256), 0, st, g);
    else hipLaunchKernelGGL((gemm_f64_kernel<T, GK, 1, 1>), grid, dim3(256), 0, st, g);
}

// 64 x 64 tiles carry twice the arithmetic per byte fetched, 32 x 32 ones fill
// the chip earlier and leave a shorter tail.  Measured, us (64, 32): L^-1 h at
// N = 1024: 49, 32; 2112: 175, 189; 4096: 1135, 1229; 7040: 5442, 7696.  With
// half the tiles and the longest k ranges on the few full columns the tail
// weighs more: W L^-T at 2112: 181, 84; 4096: 657, 531; 7040: 1883, 2417; and
// on a short k (rank 256 on the lower tiles, 4096: 131, 113; 7040: 293, 276)
// the start does.
constexpr long GEMM_TILES = 1024, GEMM_TILES_LOWER = 5120;  // whole grids of 64 x 64 tiles from which they are used
constexpr int GEMM_SHORT_K = 256;

void launch_gemm(const Gemm& g0, hipStream_t st) {
    if (g0.M <= 0 || g0.N <= 0) return;
    Gemm g = g0;
    g.c_acc = g.alpha == -1.0 && g.beta == 1.0;
    const long tiles = (long)((g.M + 63) / 64) * ((g.N + 63) / 64) * (g.batch > 0 ? g.batch : 1);
    const bool large = g.lower_only ? tiles >= GEMM_TILES_LOWER && g.K > GEMM_SHORT_K : tiles >= GEMM_TILES;
    if (large) gemm_tiles<64, 16>(g, st);
    else gemm_tiles<32, 16>(g, st);
}

// Element (r, c) of a 64 x 64 block in LDS: columns of 64, odd ones with their
// halves of 32 swapped by 16s, so that a 16 x 4 MFMA operand is read without
// bank conflicts.
__device__ __forceinline__ int blk_at(int r, int c) { return c * TILE + (r ^ ((c & 1) << 4)); }

// 16 x 16 x 16 product of two sub-blocks held in LDS (A: rows ar.., columns ac..;
// B: rows br.., columns bc..), added to acc in the plain layout (result v of
// lane l: row l/16 + 4v, column l%16), which is also the layout of a B operand:
// a product can be multiplied from the left by another without leaving the
// registers (blk_mul_reg).
__device__ __forceinline__ void blk_mul(v4d& acc, const double* A, int ar, int ac, const double* B, int br, int bc,
                                        int lane) {
    const int i = lane & 15, k = lane >> 4;
#pragma unroll
    for (int ks = 0; ks < 16; ks += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[blk_at(ar + i, ac + ks + k)], B[blk_at(br + ks + k, bc + i)], acc, 0,
                                                   0, 0);
}
__device__ __forceinline__ void blk_mul_reg(v4d& acc, const double* A, int ar, int ac, v4d b, int lane) {
    const int i = lane & 15, k = lane >> 4;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[blk_at(ar + i, ac + 4 * ks + k)], b[ks], acc, 0, 0, 0);
}

__device__ __forceinline__ double lane_value(double x, int l) {  // x of lane l (uniform), to a scalar register pair
    const long u = __double_as_longlong(x);
    const unsigned lo = __builtin_amdgcn_readlane((int)u, l), hi = __builtin_amdgcn_readlane((int)(u >> 32), l);
    return __longlong_as_double((long)(((unsigned long)hi << 32) | lo));
}

// sqrt(d) and its reciprocal for a normal d > 0 by Goldschmidt's coupled
// iteration from the hardware's estimate, with one residual correction of the
// root: both are good to an ulp.
__device__ __forceinline__ void root_and_inverse(double d, double& root, double& inv) {
    const double y = __builtin_amdgcn_rsq(d);
    double g = d * y, h = 0.5 * y;
    double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    root = fma(fma(-g, g, d), h, g);
    inv = 2.0 * h;
}
__device__ __forceinline__ double quotient(double a, double b, double binv) {  // a / b, 1/b known to an ulp
    const double q = a * binv;
    return fma(fma(-q, b, a), binv, q);
}

// inverse of the lower triangular 16 x 16 sub-block at (b0, b0) of L, column
// `lane` of it by forward substitution
__device__ __forceinline__ void invert_16(const double* L, const double* rinv, double* X, int b0, int lane) {
    if (lane >= 16) return;
    double x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        double v = i == lane ? 1.0 : 0.0;
#pragma unroll
        for (int k = 0; k < i; ++k) v = fma(-L[blk_at(b0 + i, b0 + k)], x[k], v);
        x[i] = quotient(v, L[blk_at(b0 + i, b0 + i)], rinv[b0 + i]);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) X[blk_at(b0 + i, b0 + lane)] = x[i];
}

// Block b of a panel that starts at block p0: take the panel's earlier columns
// off the 64 x 64 diagonal block (j0 = 64 b), factor it in place (lower) and
// write its inverse to Dinv[b].  One workgroup of 10 waves; bound by the serial
// chain of 64 columns, so that chain is kept short:
//   wave 0 factors 16 columns at a time with the 64 rows as its lanes and the 16
//   columns in registers: a column costs one root (root_and_inverse), one
//   quotient and, per later column, a scalar broadcast (v_readlane) and an fma;
//   the rank-16 update of the rest is one 16 x 16 MFMA block per wave;
//   while wave 0 is at columns 16 p .., wave 1 inverts diagonal sub-block p - 1
//   and wave 2 forms the (1, 0) block of the inverse; after the last columns the
//   remaining blocks follow, X_IJ = -X_II (L_IJ X_JJ ..), T = L X formed while
//   the last sub-block is inverted, products chained in registers.
// The first non-positive pivot is reported as in LAPACK's potrf (1-based).
__global__ __launch_bounds__(640) void potrf_diag_kernel(double* A, int ld, int p0, int b, double* Dinv, int* info) {
    __shared__ double Ls[TILE * TILE];
    __shared__ double Xs[TILE * TILE];
    __shared__ double rinv[TILE];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lr = lane & 15, lk = lane >> 4;
    const int j0 = b * TILE;
    int bad = 0;  // wave 0: first bad column + 1
    if (w < 10) {  // lower sub-blocks (I, J), minus the products of the panel's earlier columns
        const int I = w >= 6 ? 3 : w >= 3 ? 2 : w >= 1 ? 1 : 0, J = w - I * (I + 1) / 2;
        const double* D = A + (j0 + 16 * I + lr) + (long)ld * (j0 + 16 * J + lk);
        v4d acc;
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[v] = D[(long)ld * (4 * v)];
        for (int k0 = p0 * TILE; k0 < j0; k0 += TILE) {
            const double* LI = A + (j0 + 16 * I + lr) + (long)ld * (k0 + lk);
            const double* LJ = A + (j0 + 16 * J + lr) + (long)ld * (k0 + lk);
            double a[16], c[16];
#pragma unroll
            for (int ks = 0; ks < 16; ++ks) {
                a[ks] = LI[(long)ld * (4 * ks)];
                c[ks] = LJ[(long)ld * (4 * ks)];
            }
            __builtin_amdgcn_sched_barrier(0);  // every load is issued before the first product waits
#pragma unroll
            for (int ks = 0; ks < 16; ++ks) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(c[ks], -a[ks], acc, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) Ls[blk_at(16 * I + lr, 16 * J + lk + 4 * v)] = acc[v];
    }
    for (int e = t; e < TILE * TILE; e += 640) Xs[e] = 0.0;
    __syncthreads();
    for (int p = 0; p < 4; ++p) {
        const int k0 = 16 * p;
        if (w == 0) {
            const int row = (lane + k0) & 63;  // lanes 0..15: the diagonal sub-block; rows above it wrap to the last lanes
            double a[16], piv = 1.0, ri = 1.0;
            int ln = lane;
            asm volatile("" : "+v"(ln));  // keeps the 16 lane masks below from living in scalar registers throughout
#pragma unroll
            for (int c = 0; c < 16; ++c) a[c] = Ls[blk_at(row, k0 + c)];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const double d = lane_value(a[j], j);
                double sd, inv;
                root_and_inverse(d > 0.0 ? d : 1.0, sd, inv);
                const double l = ln == j ? sd : quotient(a[j], sd, inv);
                piv = ln == j ? d : piv;
                ri = ln == j ? inv : ri;
                a[j] = l;
#pragma unroll
                for (int c = j + 1; c < 16; ++c) a[c] = fma(-l, lane_value(l, c), a[c]);
            }
            const unsigned long long failed = __ballot(lane < 16 && !(piv > 0.0));
            if (failed && !bad) bad = k0 + __ffsll(failed);
            if (lane < 16) rinv[k0 + lane] = ri;
#pragma unroll
            for (int c = 0; c < 16; ++c) Ls[blk_at(row, k0 + c)] = a[c];
        } else if (w == 1 && p > 0) {
            invert_16(Ls, rinv, Xs, k0 - 16, lane);
        } else if (w == 2 && p == 3) {  // X_10 = -X_11 (L_10 X_00)
            v4d T = {0.0, 0.0, 0.0, 0.0}, X = {0.0, 0.0, 0.0, 0.0};
            blk_mul(T, Ls, 16, 0, Xs, 0, 0, lane);
            blk_mul_reg(X, Xs, 16, 16, T, lane);
#pragma unroll
            for (int v = 0; v < 4; ++v) Xs[blk_at(16 + lk + 4 * v, lr)] = -X[v];
        }
        __syncthreads();
        const int n2 = 3 - p;  // sub-block rows below
        if (w < n2 * (n2 + 1) / 2) {
            const int i2 = w >= 3 ? 2 : w >= 1 ? 1 : 0, I = p + 1 + i2, J = p + 1 + w - i2 * (i2 + 1) / 2;
            v4d acc;
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[v] = Ls[blk_at(16 * I + lr, 16 * J + lk + 4 * v)];
#pragma unroll
            for (int ks = 0; ks < 16; ks += 4)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(Ls[blk_at(16 * J + lr, k0 + ks + lk)],
                                                           -Ls[blk_at(16 * I + lr, k0 + ks + lk)], acc, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) Ls[blk_at(16 * I + lr, 16 * J + lk + 4 * v)] = acc[v];
        }
        __syncthreads();
    }
    // waves 4..7: T_2J, T_3J = sum_K L_IK X_KJ over K = J..1 for the lower left
    // 32 x 32 of the inverse; wave 1 inverts the last sub-block meanwhile, and
    // wave 0 then closes X_32
    v4d T2 = {0.0, 0.0, 0.0, 0.0}, T3 = {0.0, 0.0, 0.0, 0.0};
    const int J = w & 1, low = (w >> 1) & 1;  // waves 4..7: block (2 + low, J)
    if (w == 1) {
        invert_16(Ls, rinv, Xs, 48, lane);
    } else if (w >= 4 && w < 8) {
        for (int K = J; K < 2; ++K) {
            blk_mul(T2, Ls, 32, 16 * K, Xs, 16 * K, 16 * J, lane);
            if (low) blk_mul(T3, Ls, 48, 16 * K, Xs, 16 * K, 16 * J, lane);
        }
    }
    v4d T32 = {0.0, 0.0, 0.0, 0.0};
    if (w == 0) blk_mul(T32, Ls, 48, 32, Xs, 32, 32, lane);
    __syncthreads();
    if (w == 0) {
        v4d X = {0.0, 0.0, 0.0, 0.0};
        blk_mul_reg(X, Xs, 48, 48, T32, lane);
#pragma unroll
        for (int v = 0; v < 4; ++v) Xs[blk_at(48 + lk + 4 * v, 32 + lr)] = -X[v];
    }
    __syncthreads();
    if (w >= 4 && w < 8) {
        v4d X = {0.0, 0.0, 0.0, 0.0};
        blk_mul_reg(X, Xs, 32 + 16 * low, 32, T2, lane);
        if (low) blk_mul_reg(X, Xs, 48, 48, T3, lane);
#pragma unroll
        for (int v = 0; v < 4; ++v) Xs[blk_at(32 + 16 * low + lk + 4 * v, 16 * J + lr)] = -X[v];
    }
    __syncthreads();
    for (int e = t; e < TILE * TILE; e += 640) {
        const int r = e % TILE, c = e / TILE;
        A[(long)(j0 + r) + (long)ld * (j0 + c)] = r >= c ? Ls[blk_at(r, c)] : 0.0;
        Dinv[(long)b * TILE * TILE + e] = r >= c ? Xs[blk_at(r, c)] : 0.0;
    }
    if (t == 0 && bad && *info == 0) *info = j0 + bad;
}

// The column below diagonal block b of a panel that starts NK blocks earlier:
// A_ib <- (A_ib - sum_k L_ik L_bk^T) L_bb^-T over the panel's columns k before
// b.  A workgroup has 16 rows and its wave w the columns 16 w .. of the block;
// all operands come straight from memory in MFMA layout and are in flight
// together, so a launch costs one latency plus 16 (NK + 1) MFMA.  Bound by
// that latency: rest / 16 workgroups (252 at ld = 4096) of at most 64 MFMA.
template <int NK>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 2))) void chol_column_kernel(double* A, int ld, int b, const double* Dinv) {
    __shared__ double Ts[TILE * 16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
    const int j0 = b * TILE, i0 = j0 + TILE + 16 * blockIdx.x;
    double* X = A + (i0 + lr) + (long)ld * (j0 + 16 * w + lk);  // value v: column + 4 v
    const double* Di = Dinv + (long)b * TILE * TILE + (16 * w + lr) + TILE * lk;
    v4d acc;
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = X[(long)ld * (4 * v)];
    double a[16 * NK + 1], c[16 * NK + 1], di[16];
#pragma unroll
    for (int ks = 0; ks < 16 * NK; ++ks) {
        const long col = (long)ld * (j0 - NK * TILE + 4 * ks + lk);
        a[ks] = A[(i0 + lr) + col];
        c[ks] = A[(j0 + 16 * w + lr) + col];
    }
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) di[ks] = Di[TILE * (4 * ks)];
    __builtin_amdgcn_sched_barrier(0);  // every load is issued before the first product waits
#pragma unroll
    for (int ks = 0; ks < 16 * NK; ++ks) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(c[ks], -a[ks], acc, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v) Ts[(16 * w + lk + 4 * v) * 16 + lr] = acc[v];
    __syncthreads();
    acc = (v4d){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int ks = 0; ks < 16; ++ks)  // the inverse is lower triangular: columns past 16 w + 15 are zero
        if (ks < 4 * (w + 1)) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(di[ks], Ts[(4 * ks + lk) * 16 + lr], acc, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v) X[(long)ld * (4 * v)] = acc[v];
}

// zero the blocks above the diagonal blocks (column j: rows 0 .. 64 floor(j / 64) - 1),
// once the factorization is done: they hold the upper triangle of the matrix that
// came in, and nothing reads or writes them before
__global__ void zero_upper_blocks_kernel(double* A, int ld) {
    const int j = blockIdx.x;
    const int top = (j / TILE) * TILE;
    for (int i = threadIdx.x; i < top; i += blockDim.x) A[(long)i + (long)ld * j] = 0.0;
}

// Blocked Cholesky in panels of CHOL_PANEL 64-column blocks, left-looking inside
// a panel and right-looking between panels: a block takes two launches
// (potrf_diag_kernel, chol_column_kernel), which apply the panel's earlier
// columns on the fly, and the matrix right of the panel then takes one rank-256
// update: it is read and written once per 256 columns and its GEMMs run with
// K = 256.
constexpr int CHOL_PANEL = 4;

void launch_cholesky(double* A, int ld, double* Dinv, int* info, hipStream_t st) {
    const int nb = ld / TILE;
    for (int p0 = 0; p0 < nb; p0 += CHOL_PANEL) {
        const int pe = std::min(nb, p0 + CHOL_PANEL);  // blocks p0 .. pe-1
        for (int b = p0; b < pe; ++b) {
            hipLaunchKernelGGL(potrf_diag_kernel, dim3(1), dim3(640), 0, st, A, ld, p0, b, Dinv, info);
            const dim3 grid((ld - (b + 1) * TILE) / 16), block(256);
            if (grid.x == 0) continue;
            if (b == p0) hipLaunchKernelGGL(chol_column_kernel<0>, grid, block, 0, st, A, ld, b, Dinv);
            else if (b == p0 + 1) hipLaunchKernelGGL(chol_column_kernel<1>, grid, block, 0, st, A, ld, b, Dinv);
            else if (b == p0 + 2) hipLaunchKernelGGL(chol_column_kernel<2>, grid, block, 0, st, A, ld, b, Dinv);
            else hipLaunchKernelGGL(chol_column_kernel<3>, grid, block, 0, st, A, ld, b, Dinv);
        }
        // right of the panel (lower tiles only): A33 -= L31 L31^T, K = the panel's width
        const int t0 = pe * TILE, rest = ld - t0;
        if (rest <= 0) continue;
        Gemm u{};
        u.M = rest; u.N = rest; u.K = (pe - p0) * TILE;
        u.A = A + t0 + (long)ld * (p0 * TILE); u.lda = ld;
        u.B = A + t0 + (long)ld * (p0 * TILE); u.ldb = ld; u.transB = 1;
        u.C = A + t0 + (long)ld * t0; u.ldc = ld;
        u.alpha = -1.0; u.beta = 1.0; u.lower_only = 1; u.batch = 1;
        launch_gemm(u, st);
    }
    if (nb > 1) hipLaunchKernelGGL(zero_upper_blocks_kernel, dim3(ld), dim3(256), 0, st, A, ld);
}

// L^-1 by recursive doubling over the 64 x 64 diagonal blocks (whose inverses
// Dinv the Cholesky left behind).  A node of the block hierarchy splits as
//   L = [L11 0; L21 L22]  ->  L^-1 = [X11 0; -X22 L21 X11  X22],
// and every node of one level is independent, so a level is two batched
// GEMMs (T = L21 X11 with X11 lower: k >= column; X21 = -X22 T with X22
// lower: k <= row).  A level whose last node has a short right child runs
// that node with its own sizes.  work: ld * ld / 2 doubles.
__global__ void place_diag_blocks_kernel(double* X, int ld, const double* Dinv) {
    const int b = blockIdx.x;
    for (int e = threadIdx.x; e < TILE * TILE; e += blockDim.x) {
        const int r = e % TILE, c = e / TILE;
        X[(long)(b * TILE + r) + (long)ld * (b * TILE + c)] = Dinv[(long)b * TILE * TILE + e];
    }
}
__global__ void fill_zero_kernel(double* X, long n) {
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) X[t] = 0.0;
}

static void trtri_level(const double* L, double* X, int ld, double* work, int r0, int n1, int n2, int count,
                        long stride, hipStream_t st) {
    // T (n2 x n1) = L21 X11
    Gemm g{};
    g.M = n2; g.N = n1; g.K = n1;
    g.A = L + (r0 + n1) + (long)ld * r0; g.lda = ld; g.strideA = stride;
    g.B = X + r0 + (long)ld * r0; g.ldb = ld; g.strideB = stride;
    g.C = work; g.ldc = n2; g.strideC = (long)n2 * n1;
    g.alpha = 1.0; g.beta = 0.0; g.kmode = K_FROM_COLTILE; g.batch = count;
    launch_gemm(g, st);
    // X21 = -X22 T
    Gemm h{};
    h.M = n2; h.N = n1; h.K = n2;
    h.A = X + (r0 + n1) + (long)ld * (r0 + n1); h.lda = ld; h.strideA = stride;
    h.B = work; h.ldb = n2; h.strideB = (long)n2 * n1;
    h.C = X + (r0 + n1) + (long)ld * r0; h.ldc = ld; h.strideC = stride;
    h.alpha = -1.0; h.beta = 0.0; h.kmode = K_BELOW_ROWTILE; h.batch = count;
    launch_gemm(h, st);
}

void launch_trtri_lower(const double* L, double* X, const double* Dinv, int ld, double* work, hipStream_t st) {
    const long n = (long)ld * ld;
    hipLaunchKernelGGL(fill_zero_kernel, dim3(4096), dim3(256), 0, st, X, n);
    const int nb = ld / TILE;
    hipLaunchKernelGGL(place_diag_blocks_kernel, dim3(nb), dim3(256), 0, st, X, ld, Dinv);
    for (int hb = 1; hb < nb; hb *= 2) {  // child size in blocks
        const int b = hb * TILE;
        const int full = nb / (2 * hb);
        const long stride = 2L * b * (ld + 1);
        if (full > 0) trtri_level(L, X, ld, work, 0, b, b, full, stride, st);
        const int rem = nb - full * 2 * hb;
        if (rem > hb) trtri_level(L, X, ld, work, full * 2 * b, b, (rem - hb) * TILE, 1, 0, st);
    }
}

__global__ void symmetrize_from_lower_kernel(double* A, int ld) {
    // tile-transposing copy of the strictly lower part into the upper part
    __shared__ double tile[32][33];
    const int bx = blockIdx.x, by = blockIdx.y;
    if (bx > by) return;  // source tile (row block by, col block bx) in the lower part
    const int tx = threadIdx.x, ty = threadIdx.y;
    for (int r = ty; r < 32; r += blockDim.y) {
        const int i = by * 32 + r, j = bx * 32 + tx;
        tile[r][tx] = A[(long)i + (long)ld * j];
    }
    __syncthreads();
    for (int r = ty; r < 32; r += blockDim.y) {
        // destination (row j, col i) with j = bx*32 + r, i = by*32 + tx
        const int j = bx * 32 + r, i = by * 32 + tx;
        if (i > j) A[(long)j + (long)ld * i] = tile[tx][r];
    }
}

void launch_symmetrize_from_lower(double* A, int ld, hipStream_t st) {
    const int nb = ld / 32;
    hipLaunchKernelGGL(symmetrize_from_lower_kernel, dim3(nb, nb), dim3(32, 8), 0, st, A, ld);
}

__global__ void copy_kernel(const double* s, double* d, long n) {
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < n; t += (long)gridDim.x * blockDim.x) d[t] = s[t];
}
void launch_copy_matrix(const double* src, double* dst, long n, hipStream_t st) {
    hipLaunchKernelGGL(copy_kernel, dim3(4096), dim3(256), 0, st, src, dst, n);
}

// S <- identity, h <- 0 over the whole ld x ld buffer (the host block is copied in afterwards).
__global__ void identity_pad_kernel(double* S, double* h, int ld) {
    const long total = (long)ld * ld;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
        const int i = (int)(t % ld), j = (int)(t / ld);
        S[t] = i == j ? 1.0 : 0.0;
        h[t] = 0.0;
    }
}
void launch_identity_pad(double* S, double* h, int N, int ld, hipStream_t st) {
    (void)N;
    hipLaunchKernelGGL(identity_pad_kernel, dim3(4096), dim3(256), 0, st, S, h, ld);
}

// rows x cols column-major block between two pitches (rows as lanes: coalesced
// both ways; HBM-bound)
__global__ __launch_bounds__(256) void repitch_kernel(double* __restrict__ dst, long ldd,
                                                      const double* __restrict__ src, long lds, int rows) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < rows) dst[ldd * blockIdx.y + i] = src[lds * blockIdx.y + i];
}
void launch_repitch(double* dst, long ldd, const double* src, long lds, int rows, int cols, hipStream_t st) {
    constexpr int MAX_Y = 32768;  // columns per launch (grid limit)
    for (int c = 0; c < cols; c += MAX_Y)
        hipLaunchKernelGGL(repitch_kernel, dim3((rows + 255) / 256, std::min(cols - c, MAX_Y)), dim3(256), 0, st,
                           dst + ldd * c, ldd, src + lds * c, lds, rows);
}

}  // namespace dh

// The k loop of the FP64 products: a T x T tile of opA(A) opB(B) over a range
// of k, for the dense algebra (dense.hip) and for the operator on many columns
// (cheb.hip).
//
// 256 threads = 4 waves in a 2 x 2 arrangement, each wave a T/2 x T/2 quadrant
// of 16 x 16 MFMA blocks (v_mfma_f64_16x16x4f64: lane l holds A[l%16][l/16] and
// B[l/16][l%16]; result v of lane l is D[l/16 + 4v][l%16]).  The MFMA is issued
// with the operands swapped (D^T = B^T A^T), so a lane's four results lie in
// four columns and each column's 16 rows are contiguous in a column-major C.
//
// Bound: the matrix cores (64 cycles per instruction and SIMD).  A GK-deep k
// stage is double-buffered in LDS; the stage after next is fetched into
// registers while the current one is multiplied.  A stage is one scheduling
// region in which fetches, LDS writes of the next stage and operand reads go
// between the products (gemm_order): issued in blocks instead, they leave the
// matrix cores idle, since a wave issues in order and a running product hides 64
// cycles only.  The LDS rows are XOR-swizzled (gemm_sw) instead of padded:
// operand reads (16 rows x 4 k), row-wise stores and k-wise stores (transposed
// operands) are all free of bank conflicts.  Full products of 4096, T = 64,
// three workgroups a CU: 68 TFLOP/s; 55 with the memory instructions in blocks,
// 75 for the bare products.
#pragma once
#include "common.hpp"

namespace dh {

__device__ __forceinline__ int gemm_sw(int k) { return ((k & 1) << 4) | (k & 14); }

// Issue order of one k stage: the operand reads of the next products, the
// fetches for the stage after next and the writes of the next stage go between
// the products, a few per product, so that each is issued in the shadow of a
// running one.
template <int I, int NM, int NR, int NV, int NW, int RP>
__device__ __forceinline__ void gemm_order() {
    if constexpr (I < NM) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // a product
        constexpr int reads = (NR - RP) * (I + 1) / NM - (NR - RP) * I / NM;
        if constexpr (reads > 0) __builtin_amdgcn_sched_group_barrier(0x100, reads, 0);
        constexpr int loads = NV * (I + 1) / NM - NV * I / NM;
        if constexpr (loads > 0) __builtin_amdgcn_sched_group_barrier(0x020, loads, 0);
        constexpr int writes = NW * (I + 1) / NM - NW * I / NM;
        if constexpr (writes > 0) __builtin_amdgcn_sched_group_barrier(0x200, writes, 0);
        gemm_order<I + 1, NM, NR, NV, NW, RP>();
    }
}

// acc += A B over k in [klo, khi).  A points to the tile's first row at k = 0
// (k contiguous with TA, else rows contiguous, EA = float is widened), B to its
// first column (columns contiguous with TB, else k contiguous); na and nb rows
// and columns of the tile exist: those past them are read from the last one.
// keep(i, k) says for MASKED products which elements of A count (i within the
// tile); bcol(j) is the place of column j of a TB tile, in elements from B.  Every thread of the workgroup calls it; it ends with a barrier.
template <int T, int GK, int TA, int TB, bool MASKED, typename EA, typename Keep, typename BCol>
__device__ __forceinline__ void gemm_accumulate(v4d (&acc)[T / 32][T / 32], const EA* A, long lda, int na,
                                                const double* B, long ldb, int nb, int klo, int khi,
                                                double (*As)[GK * T], double (*Bs)[GK * T], const Keep& keep,
                                                const BCol& bcol) {
    constexpr int MB = T / 32;        // 16 x 16 blocks of a wave per direction
    constexpr int NL = GK * T / 256;  // values a thread fetches per operand and stage
    constexpr int EB = (int)sizeof(EA);
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int wi = (w >> 1) * (T / 2), wj = (w & 1) * (T / 2);
    const int lr = lane & 15, lk = lane >> 4;
    // value r of this thread: row (column) ia (jb), depth ka (kb) of the stage
    auto ia = [&](int r) { return TA ? t / GK + (256 / GK) * r : t % T; };
    auto ka = [&](int r) { return TA ? t % GK : t / T + (256 / T) * r; };
    auto jb = [&](int r) { return TB ? t % T : t / GK + (256 / GK) * r; };
    auto kb = [&](int r) { return TB ? t / T + (256 / T) * r : t % GK; };
    const long sa = TA ? 1 : lda, sb = TB ? ldb : 1;  // strides of one k
    int oa[NL], ob[NL];                               // byte offsets from the stage's first k
#pragma unroll
    for (int r = 0; r < NL; ++r) {
        oa[r] = EB * (min(ia(r), na - 1) * (TA ? (int)lda : 1) + ka(r) * (int)sa);
        ob[r] = 8 * ((TB ? bcol(min(jb(r), nb - 1)) : min(jb(r), nb - 1) * (int)ldb) + kb(r) * (int)sb);
    }
    const int ns = khi > klo ? (khi - klo + GK - 1) / GK : 0;  // stages; a last one that is not whole starts
    const int skip = ns * GK - (khi - klo);                    // earlier, its first `skip` depths count as zero
    const EA* pa = A + sa * klo;  // the next stage to fetch
    const double* pb = B + sb * klo;
    int kw = klo;                 // first k of the next stage to write to LDS
    double rb[2][NL];
    EA ra[2][NL];
    auto rsrc = [](const void* base) { return __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0x7fffffff, 0x00020000); };
    auto at_a = [&](const EA* base, int o) -> EA {  // scalar base, 32-bit lane offset
        if constexpr (EB == 8) return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc(base), o, 0, 0));
        else return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc(base), o, 0, 0));
    };
    auto at_b = [&](const double* base, int o) {
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc(base), o, 0, 0));
    };
    auto gload = [&](int q) {
#pragma unroll
        for (int r = 0; r < NL; ++r) {
            ra[q][r] = at_a(pa, oa[r]);
            rb[q][r] = at_b(pb, ob[r]);
        }
        pa += GK * sa;
        pb += GK * sb;
    };
    auto put = [&](int q, int r, bool za, double va, bool zb, double vb) {
        if (MASKED) za = za || !keep(ia(r), kw + ka(r));
        As[q][ka(r) * T + (ia(r) ^ gemm_sw(ka(r)))] = za ? 0.0 : va;
        Bs[q][kb(r) * T + (jb(r) ^ gemm_sw(kb(r)))] = zb ? 0.0 : vb;
    };
    auto swrite = [&](int q, int z) {  // the first z depths as zero
        kw -= z;
#pragma unroll
        for (int r = 0; r < NL; ++r) put(q, r, ka(r) < z, (double)ra[q][r], kb(r) < z, rb[q][r]);
        kw += GK;
    };
    auto multiply = [&](int q) {
#pragma unroll
        for (int ks = 0; ks < GK; ks += 4) {
            double av[MB], bv[MB];
            const int k = ks + lk, x = gemm_sw(k);
#pragma unroll
            for (int a = 0; a < MB; ++a) av[a] = As[q][k * T + ((wi + a * 16 + lr) ^ x)];
#pragma unroll
            for (int b = 0; b < MB; ++b) bv[b] = Bs[q][k * T + ((wj + b * 16 + lr) ^ x)];
#pragma unroll
            for (int a = 0; a < MB; ++a)
#pragma unroll
                for (int b = 0; b < MB; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(bv[b], av[a], acc[a][b], 0, 0, 0);
        }
    };
    if (ns > 1) {
        gload(0);
        if (ns == 2) pa -= sa * skip, pb -= sb * skip;
        gload(1);
        swrite(0, 0);
    } else if (ns == 1) {  // one stage: depths past the end are read from the last one and count as zero
        const int last = khi - 1 - klo;
#pragma unroll
        for (int r = 0; r < NL; ++r) {
            const int da = max(ka(r) - last, 0), db = max(kb(r) - last, 0);
            put(0, r, da > 0, (double)at_a(pa, oa[r] - EB * da * (int)sa), db > 0, at_b(pb, ob[r] - 8 * db * (int)sb));
        }
    }
    __syncthreads();
    // stage st is in LDS buffer q, st + 1 in registers 1 - q, st + 2 is asked for
    constexpr int NM = MB * MB * GK / 4, NR = 2 * MB * GK / 4, RP = 4 * MB;  // reads ahead: two k steps of 4
    int st = 0;
    auto whole = [&](int q) {
        gload(q);
        multiply(q);
        swrite(1 - q, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, RP, 0);
        gemm_order<0, NM, NR, 2 * NL, 2 * NL, RP>();
        __syncthreads();
    };
    for (; st + 4 < ns; st += 2) {
        whole(0);
        whole(1);
    }
    auto rest = [&](int q) {
        if (st + 2 < ns) {
            if (st + 3 == ns) pa -= sa * skip, pb -= sb * skip;
            gload(q);
        }
        multiply(q);
        if (st + 1 < ns) swrite(1 - q, st + 2 == ns ? skip : 0);
        __syncthreads();
        ++st;
    };
    while (st < ns) {
        rest(0);
        if (st < ns) rest(1);
    }
}

}  // namespace dh

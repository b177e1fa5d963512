// A whole Chebyshev series in one launch, with the operator resident on the chip.
//
// A term of the recurrence reads all of H_orth, which does not change within a
// series.  Launched term by term (cheb.hip), a term is bound by that read: at
// N = 4096 and R = 4 columns the symmetric half of H (68 MB) and the partial
// sums of its column products take 21 us per term.  The register files (128 MB)
// and LDS (40 MB) of the 256 CUs together hold the whole of a 4096 x 4096 H
// (134 MB), so this kernel loads H once, keeps each workgroup's rows of it in
// registers and LDS, and runs every term of the series with nothing read from
// memory but the previous term's vectors, which the workgroups exchange
// through global memory behind one flag per workgroup and term.  Per term, one
// launch per term against this kernel: N = 4096, R = 4: 21.6 -> 6.9 us; N =
// 2048: 10.3 -> 4.7 us (R = 4), 17 -> 5.5 us (R = 8); N = 416: 7.2 -> 2.9 us.
// At N = 4096 a term is now 3.4 us of matrix-core time, about 1.4 us of waiting
// for the other workgroups' flags and 1.5 us of latencies (first loads of x,
// the sum over the waves, the store); at N = 416 it is latency alone.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace dh {

// Work split: workgroup b owns RB = 4 RG consecutive rows; its 8 waves split
// the columns (the reduction index) into 8 ranges of `groups` 16-column groups.
// A group's products are FP64 MFMA 4x4x4 in 4 blocks (lanes A: 16k + 4b + i,
// B: 16k + 4b + j, D: 16i + 4b + j) with block b taking columns 4b..4b+3 of the
// group, so a B operand (x) feeds every row group without replication: lane
// 16k + 4b + j loads x[16g + 4b + k][j], 16 bytes (re, im) per lane, 1 KB
// contiguous per wave.  A operands (H) stay in the lane's registers, up to what
// 256 registers hold beside the products (23 groups at R = 4), and in LDS from
// there on.  At R = 4 a group is 8 MFMAs of 16 cycles on one load; N = 4096: 32
// groups per wave, 3.4 us of matrix-core time per term.
//
// Exchange: T_k goes to slot k % slots of a ring with stores that bypass the
// XCD's L2 (device scope); the storing wave waits for them and then raises the
// workgroup's flag to k + 1.  A wave of term k + 1 waits for the flags of the
// rows it reads only.  The data is read with ordinary cached loads (each XCD
// fetches a slot once, its other CUs hit L2): a slot's lines are not in L1 or
// L2 from an earlier term because the ring's addresses are read once per lap,
// and every wave invalidates both (device-scope acquire) when it starts a lap.
// A slot is overwritten `slots` terms later: a workgroup that writes T_{k+1}
// has seen every flag of term k, so every wave is past reading T_{k-1}.
//
// All workgroups must be on the chip at once, so the launch is cooperative,
// and every wait is bounded (wall clock): a wave that runs out of time stops
// waiting for good, the kernel drains, and its workgroup's accumulators are
// written as NaN, which the caller's norm check turns into a repeat of the
// step with one launch per term.
constexpr int RS_WAVES = 8;
constexpr int RS_THREADS = RS_WAVES * 64;
// Copies of the flags, each polled by every RS_COPIES-th workgroup: with one
// copy the 2048 waves' polls of the same few lines queue up at one memory
// channel (a term at N = 4096, R = 4: 8.9 us with one copy, 7.6 with 8).
constexpr int RS_COPIES = 16;
constexpr int RS_NQ = (MULTI_MAX + RS_WAVES - 1) / RS_WAVES;  // accumulators per wave
constexpr unsigned long long RS_WAIT_TICKS = 200000000ull;    // 2 s of the 100 MHz wall clock
constexpr int AUX_DEVICE_SCOPE = 16;                          // buffer store: sc1

typedef int v4i __attribute__((ext_vector_type(4)));
// the coefficient table does not change during the launch: constant address
// space, so wave-uniform reads go to scalar registers
typedef const __attribute__((address_space(4))) double* rs_const;
__device__ __forceinline__ cplx rs_coef(const cplx* p) {
    const rs_const d = (rs_const)(p);
    return cplx{d[0], d[1]};
}

template <int CTRL>
__device__ __forceinline__ double rs_dpp(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
// sum over the four blocks (lanes 4 apart of a row of 16)
__device__ __forceinline__ double rs_block_sum(double v) {
    const double z = v + rs_dpp<0x128>(v);  // row rotate 8
    return z + rs_dpp<0x124>(z);            // row rotate 4
}

// LDS contents of the workgroup are visible to all its waves past this point
// (global stores may still be in flight, unlike with __syncthreads)
__device__ __forceinline__ void rs_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// RC: passes of 4 complex columns over H per term (1: R <= 4, 2: R <= 8), a lane's
// x being one complex column; 0: one pass of up to 4 real columns (R <= 2).
// NT: groups per wave, a compile-time count so that the loads of x run ahead of
// the products through the whole unrolled sequence.
constexpr int rs_most(int rc) { return rc == 0 ? 24 : rc == 1 ? 23 : 20; }
template <int RG, int NT, int RC>
__global__ __launch_bounds__(RS_THREADS, 2) void resident_series_kernel(const ResidentArgs a) {
    constexpr int NREG = RG == 4 && NT > rs_most(RC) ? rs_most(RC) : NT, NL = NT - NREG;
    constexpr bool PAIR = RC > 0;
    constexpr int RB = 4 * RG, np = PAIR ? RC : 1;
    // x loads in flight per wave: what the registers beside H allow
    constexpr int DEPTH = std::min(NT, RG == 2 ? 6 : NREG > 20 ? 4 : NREG > 12 ? 6 : 8);
    using xv_t = typename std::conditional<PAIR, double2, double>::type;
    extern __shared__ double smem[];
    const int R = a.R;
    constexpr int n = NT;
    double* const hs = smem;                                       // [NL][8][RG][64]
    cplx* const part = reinterpret_cast<cplx*>(hs + NL * RS_WAVES * RG * 64);  // [np][8][RB * 4]
    cplx* const ts = part + np * RS_WAVES * RB * 4;                // [3][RB * R]: the last three terms' own rows
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lk = lane >> 4, lb = (lane >> 2) & 3, lj = lane & 3;
    const int N = a.N, ld = a.ld;
    const int r0 = blockIdx.x * RB, k0 = w * n * 16;
    const bool active = k0 < ld;      // this wave has columns
    const int E = RB * R;             // own elements

    // H: rows r0 + 4 rg + lj, columns k0 + 16 g + 4 lb + lk; ld is a multiple of
    // 64, so a group lies inside the matrix or past it (zero) as a whole
    const int ng = active ? min(n, (ld - k0) / 16) : 0;
    double h[NREG][RG];
    const double* const hcol = a.H + (long)ld * (r0 + lj) + 4 * lb + lk;
    auto hval = [&](int g, int rg) {
        const double v = hcol[(long)ld * (4 * rg) + (g < ng ? k0 + 16 * g : 0)];
        return g < ng ? v : 0.0;
    };
#pragma unroll
    for (int g = 0; g < NREG; ++g)
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) h[g][rg] = hval(g, rg);
#pragma unroll 1
    for (int g = 0; g < NL; ++g)
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) hs[((g * RS_WAVES + w) * RG + rg) * 64 + lane] = hval(NREG + g, rg);

    // the wave's accumulators: q = w + 8 v, elements lane + 64 u of the workgroup's rows
    constexpr int NE = (RB * (PAIR ? 4 * RC : 2) + 63) / 64;
    cplx acc[RS_NQ][NE];
    int kq[RS_NQ];
#pragma unroll
    for (int v = 0; v < RS_NQ; ++v) {
        const int q = w + RS_WAVES * v;
        kq[v] = q < a.m ? (a.kq ? __builtin_amdgcn_readfirstlane(a.kq[q]) : a.K) : -1;
    }
    const __amdgpu_buffer_rsrc_t ring =
        __builtin_amdgcn_make_buffer_rsrc(a.ring, 0, (int)(a.slots * a.slot_bytes), 0x00020000);
    // element e's place in a slot: its row-major position
    auto publish = [&](int e, cplx T, int slot) {
        v4i bits;
        bits[0] = __double2loint(T.re);
        bits[1] = __double2hiint(T.re);
        bits[2] = __double2loint(T.im);
        bits[3] = __double2hiint(T.im);
        __builtin_amdgcn_raw_buffer_store_b128(bits, ring, (r0 * R + e) * 16, slot * a.slot_bytes, AUX_DEVICE_SCOPE);
    };
    auto raise = [&](unsigned v) {  // after this wave's stores have arrived
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (lane < RS_COPIES)
            __hip_atomic_store(a.flags + lane * (int)gridDim.x + blockIdx.x, v, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    };

    // T_0 = phi (rows >= N as zero)
    if (w == 0) {
        for (int e = lane; e < E; e += 64) {
            const int row = r0 + e / R;
            const cplx T = row < N ? a.phi[(long)r0 * R + e] : cplx{0.0, 0.0};
            publish(e, T, 0);
            ts[e] = T;
        }
        raise(1u);
    }
    rs_lds_barrier();
#pragma unroll
    for (int v = 0; v < RS_NQ; ++v)
        if (kq[v] >= 0) {
            const cplx c0 = rs_coef(a.coef + (long)(w + RS_WAVES * v) * a.coef_stride);
#pragma unroll
            for (int u = 0; u < NE; ++u)
                if (lane + 64 * u < E) acc[v][u] = cmul(c0, ts[lane + 64 * u]);
        }

    // this lane's x of the wave's group g: row k0 + 16 g + 4 lb + lk, column
    // 4 p + lj (columns past the last read it again; their sums are not kept).
    // Groups past ld read the last one (their H is zero).
    const int C2 = PAIR ? R : 2 * R;  // x values per row
    const int xbytes = (int)sizeof(xv_t);
    const int gstride = 16 * R * 16;
    // flags of the rows this wave reads
    const int f0 = k0 / RB, nf = active ? (min(k0 + 16 * n, ld) + RB - 1) / RB - f0 : 0;
    const unsigned* const myflag = a.flags + (int)(blockIdx.x % RS_COPIES) * (int)gridDim.x + f0 + min(lane, max(nf - 1, 0));
    bool dead = false;
    const double a1 = 1.0 / a.r, b1 = -a.c / a.r;
    const int K = max(a.K, 1);
    for (int k = 1; k <= K; ++k) {
        cplx ck[RS_NQ];
#pragma unroll
        for (int v = 0; v < RS_NQ; ++v)
            if (k <= kq[v]) ck[v] = rs_coef(a.coef + (long)(w + RS_WAVES * v) * a.coef_stride + k);
        if (active) {
            if (!dead) {
                unsigned long long t0 = 0;
                for (int spin = 0;; ++spin) {
                    const unsigned v = __hip_atomic_load(myflag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (__ballot((int)(v - (unsigned)k) < 0) == 0) break;
                    if ((spin & 255) == 255) {
                        const unsigned long long now = wall_clock64();
                        if (t0 == 0) t0 = now;
                        else if (now - t0 > RS_WAIT_TICKS) {
                            dead = true;
                            break;
                        }
                    }
                }
            }
            asm volatile("" ::: "memory");
            const int slot = (k - 1) % a.slots;
            if (slot == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            // PT passes together (their loads and products interleave), where the
            // registers allow
            constexpr int PT = RG == 4 ? 1 : np;
#pragma unroll 1
            for (int p0 = 0; p0 < np; p0 += PT) {
                int xoff[PT];
#pragma unroll
                for (int p = 0; p < PT; ++p)
                    xoff[p] = ((k0 + 4 * lb + lk) * C2 + min(4 * (p0 + p) + lj, C2 - 1)) * xbytes;
                const int soff = slot * a.slot_bytes;
                auto xload = [&](int g, int p) -> xv_t {
                    const int so = soff + min(g, max(ng, 1) - 1) * gstride;
                    if constexpr (PAIR)
                        return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(ring, xoff[p], so, 0));
                    else
                        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ring, xoff[p], so, 0));
                };
                double yr[PT][RG], yi[PT][RG];
#pragma unroll
                for (int p = 0; p < PT; ++p)
#pragma unroll
                    for (int rg = 0; rg < RG; ++rg) yr[p][rg] = yi[p][rg] = 0.0;
                auto mma = [&](double hv, xv_t x, int p, int rg) {
                    if constexpr (PAIR) {
                        yr[p][rg] = __builtin_amdgcn_mfma_f64_4x4x4f64(hv, x.x, yr[p][rg], 0, 0, 0);
                        yi[p][rg] = __builtin_amdgcn_mfma_f64_4x4x4f64(hv, x.y, yi[p][rg], 0, 0, 0);
                    } else {
                        yr[p][rg] = __builtin_amdgcn_mfma_f64_4x4x4f64(hv, x, yr[p][rg], 0, 0, 0);
                    }
                };
                // step s takes register group s, and LDS group NREG + l after
                // register group NREG - NL + l, whose products cover its LDS reads
                constexpr int RONLY = NREG - NL;
                auto group = [](int st) {
                    return st < RONLY ? st : (st - RONLY) % 2 == 0 ? RONLY + (st - RONLY) / 2 : NREG + (st - RONLY) / 2;
                };
                xv_t xb[DEPTH][PT];
#pragma unroll
                for (int d = 0; d < DEPTH; ++d)
#pragma unroll
                    for (int p = 0; p < PT; ++p) xb[d][p] = xload(group(d), p);
                double hl[RG];
#pragma unroll
                for (int st = 0; st < NT; ++st) {
                    const int g = group(st);
                    if (g < NREG && st >= RONLY && NL > 0) {
#pragma unroll
                        for (int rg = 0; rg < RG; ++rg)
                            hl[rg] = hs[(((st - RONLY) / 2 * RS_WAVES + w) * RG + rg) * 64 + lane];
                    }
#pragma unroll
                    for (int p = 0; p < PT; ++p) {
                        const xv_t x = xb[st % DEPTH][p];
                        if (st + DEPTH < NT) xb[st % DEPTH][p] = xload(group(st + DEPTH), p);
#pragma unroll
                        for (int rg = 0; rg < RG; ++rg) mma(g < NREG ? h[g < NREG ? g : 0][rg] : hl[rg], x, p, rg);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                // lane (i, b, j) keeps row group b (b < RG): row 4 b + i, column j
#pragma unroll
                for (int p = 0; p < PT; ++p) {
                    double sr[RG], si[RG];
#pragma unroll
                    for (int rg = 0; rg < RG; ++rg) {
                        sr[rg] = rs_block_sum(yr[p][rg]);
                        si[rg] = PAIR ? rs_block_sum(yi[p][rg]) : 0.0;
                    }
                    double vr = sr[0], vi = si[0];
#pragma unroll
                    for (int rg = 1; rg < RG; ++rg) {
                        vr = lb == rg ? sr[rg] : vr;
                        vi = lb == rg ? si[rg] : vi;
                    }
                    if (lb < RG) {
                        if constexpr (PAIR) {
                            part[((p0 + p) * RS_WAVES + w) * RB * 4 + (4 * lb + lk) * 4 + lj] = cplx{vr, vi};
                        } else if (lj < 2 * R) {  // real columns: packed as R complex ones
                            reinterpret_cast<double*>(part)[w * RB * 8 + (4 * lb + lk) * 2 * R + lj] = vr;
                        }
                    }
                }
            }
        } else {
            for (int e = lane; e < np * RB * 4; e += 64) {
                const int p = e / (RB * 4), f = e % (RB * 4);
                part[(p * RS_WAVES + w) * RB * 4 + f] = cplx{0.0, 0.0};
            }
        }
        rs_lds_barrier();
        cplx* const tk = ts + (k % 3) * E;
        if (w == 0) {
            const cplx* const t1 = ts + ((k + 2) % 3) * E;
            const cplx* const t2 = ts + ((k + 1) % 3) * E;
            const double alpha = k == 1 ? a1 : 2.0 * a1, beta = k == 1 ? b1 : 2.0 * b1;
#pragma unroll
            for (int u = 0; u < NE; ++u) {
                const int e = lane + 64 * u;
                if (e < E) {
                    cplx y{0.0, 0.0};
                    const int row = e / R, col = e % R;
                    const cplx* pp = PAIR ? part + (col / 4) * RS_WAVES * RB * 4 + row * 4 + col % 4 : part + e;
#pragma unroll(RG == 4 && NREG > 16 ? 4 : RS_WAVES)
                    for (int ww = 0; ww < RS_WAVES; ++ww) {
                        y.re += pp[ww * RB * 4].re;
                        y.im += pp[ww * RB * 4].im;
                    }
                    const cplx xv = t1[e];
                    cplx T{alpha * y.re + beta * xv.re, alpha * y.im + beta * xv.im};
                    if (k > 1) {
                        const cplx x2 = t2[e];
                        T.re -= x2.re;
                        T.im -= x2.im;
                    }
                    if (k < K) publish(e, T, k % a.slots);
                    tk[e] = T;
                }
            }
            if (k < K) raise((unsigned)k + 1u);
        }
        rs_lds_barrier();
#pragma unroll
        for (int v = 0; v < RS_NQ; ++v)
            if (k <= kq[v]) {
#pragma unroll
                for (int u = 0; u < NE; ++u)
                    if (lane + 64 * u < E) {
                        const cplx add = cmul(ck[v], tk[lane + 64 * u]);
                        acc[v][u].re += add.re;
                        acc[v][u].im += add.im;
                    }
            }
    }
    // a wave that gave up waiting marks its workgroup's result
    unsigned* const gave_up = reinterpret_cast<unsigned*>(part);
    if (t == 0) *gave_up = 0u;
    rs_lds_barrier();
    if (dead) *gave_up = 1u;
    rs_lds_barrier();
    const bool bad = *gave_up != 0u;
#pragma unroll
    for (int v = 0; v < RS_NQ; ++v) {
        const int q = w + RS_WAVES * v;
        if (kq[v] >= 0) {
#pragma unroll
            for (int u = 0; u < NE; ++u) {
                const int e = lane + 64 * u;
                if (e < E && r0 + e / R < N) {
                    const cplx z = bad ? cplx{__builtin_nan(""), __builtin_nan("")} : acc[v][u];
                    a.acc[(long)q * a.acc_stride + (long)r0 * R + e] = z;
                }
            }
        }
    }
}

// ------------------------------------------------------------------ plan
// Rows per workgroup: 16 (RG = 4), which reads x least often per product; 8 for
// R > 4 while that leaves at most 256 workgroups, since both passes over H then
// run together (N = 2048, R = 8: 5.5 against 7.6 us per term; at R = 4 8 rows
// measured the same as 16).  NT: the groups a
// wave needs, rounded up to even above 8 (the surplus is zero).
struct ResidentPlan {
    int RG = 0, RC = 0, NT = 0, wgs = 0, lds = 0;
    bool ok = false;
};

static ResidentPlan resident_plan(int ld, int R, int cus) {
    ResidentPlan p;
    if (!(R >= 1 && R <= 8) || ld <= 0 || ld > 4096) return p;
    p.RC = R <= 2 ? 0 : R <= 4 ? 1 : 2;
    p.RG = p.RC == 2 && ld <= 2048 ? 2 : 4;
    p.wgs = ld / (4 * p.RG);
    const int n = (ld / 16 + RS_WAVES - 1) / RS_WAVES;
    p.NT = n <= 8 ? n : (n + 1) / 2 * 2;
    const int np = p.RC == 2 ? 2 : 1, nl = p.RG == 4 ? std::max(0, p.NT - rs_most(p.RC)) : 0;
    p.lds = nl * RS_WAVES * p.RG * 64 * 8 + np * RS_WAVES * 4 * p.RG * 4 * 16 + 3 * 4 * p.RG * R * 16;
    p.ok = p.wgs <= cus && p.lds <= 160 * 1024 && (p.RC < 2 || p.NT <= 28);
    return p;
}

bool resident_series_fits(int ld, int R, int cus) { return resident_plan(ld, R, cus).ok; }

// bytes of one ring slot, and of the flags in front of the ring
static long resident_slot_bytes(int ld, int R) { return (long)ld * R * 16; }
static long resident_flag_bytes(int ld) { return (long)RS_COPIES * (ld / 4) * 4; }

template <int RG, int NT, int RC>
static hipError_t resident_go(const ResidentArgs& a, const ResidentPlan& p, hipStream_t st) {
    const void* f = reinterpret_cast<const void*>(&resident_series_kernel<RG, NT, RC>);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, p.lds);
    if (e != hipSuccess) return e;
    ResidentArgs arg = a;
    void* params[] = {&arg};
    return hipLaunchCooperativeKernel(f, dim3(p.wgs), dim3(RS_THREADS), params, (unsigned)p.lds, st);
}

// the kernel of p.NT among LO, LO + STEP, ..., HI
template <int RG, int RC, int LO, int HI, int STEP>
static hipError_t resident_pick(const ResidentArgs& a, const ResidentPlan& p, hipStream_t st) {
    if (p.NT == LO) return resident_go<RG, LO, RC>(a, p, st);
    if constexpr (LO + STEP <= HI) return resident_pick<RG, RC, LO + STEP, HI, STEP>(a, p, st);
    return hipErrorInvalidValue;
}

static hipError_t resident_launch(const ResidentArgs& a, const ResidentPlan& p, hipStream_t st) {
    const bool few = p.NT <= 8;
    if (p.RC == 0) return few ? resident_pick<4, 0, 1, 8, 1>(a, p, st) : resident_pick<4, 0, 10, 32, 2>(a, p, st);
    if (p.RC == 1) return few ? resident_pick<4, 1, 1, 8, 1>(a, p, st) : resident_pick<4, 1, 10, 32, 2>(a, p, st);
    if (p.RG == 2) return few ? resident_pick<2, 2, 1, 8, 1>(a, p, st) : resident_pick<2, 2, 10, 16, 2>(a, p, st);
    return resident_pick<4, 2, 18, 28, 2>(a, p, st);
}

// scratch: flags, then as many ring slots as fit (at least 4)
bool launch_resident_series(ResidentArgs a, void* scratch, long scratch_bytes, int cus, hipStream_t st) {
    const ResidentPlan p = resident_plan(a.ld, a.R, cus);
    const long fb = resident_flag_bytes(a.ld), sb = resident_slot_bytes(a.ld, a.R);
    const long slots = std::min(64L, (scratch_bytes - fb) / sb);
    if (!p.ok || slots < 4 || a.m < 1 || a.m > MULTI_MAX) return false;
    a.flags = static_cast<unsigned*>(scratch);
    a.ring = static_cast<char*>(scratch) + fb;
    a.slots = (int)slots;
    a.slot_bytes = (int)sb;
    launch_zero_u32(a.flags, (int)(fb / 4), st);
    const hipError_t e = resident_launch(a, p, st);
    if (e == hipSuccess) return true;
    (void)hipGetLastError();  // not launched: the caller runs the series term by term
    return false;
}

}  // namespace dh

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
// through global memory: behind one flag per workgroup and term, or (EAGER below)
// with the data as their own flags.  Per term, one launch per term against this
// kernel: N = 4096, R = 4: 21.6 -> 6.9 us; N = 2048: 10.3 -> 4.1 us (R = 4), 17 ->
// 5.2 us (R = 8); N = 416: 7.2 -> 2.3 us.  At N = 4096 a term is now 3.4 us of
// matrix-core time, about 1.4 us of waiting for the other workgroups' flags and
// 1.5 us of latencies (first loads of x, the sum over the waves, the store); at N
// = 416 it is the latency of one exchange.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <atomic>
#include <mutex>

namespace dh {

// ------------------------------------------------------------------ cooperative launches
// One turnstile per device.  A kernel of this kind needs all its workgroups on the
// chip at once, so two of them gain nothing from overlapping, and two that held
// part of the chip each would wait for one another until their waits ran out.
// The lock is held over the launch, so that no two threads are ever inside the
// runtime's cooperative launch (nor in its first-use set-up) at the same time, and
// over the wait for another owner's launches to end; launches of one owner, which
// one thread makes, are ordered by the runtime.
namespace {
constexpr int MAX_DEVICES = 64, OWNER_STREAMS = 2;  // a context's stream and its side stream
struct Turnstile {
    std::mutex mu;
    const void* owner = nullptr;  // whose launches may be in flight; null: nobody's
    hipEvent_t done[OWNER_STREAMS] = {};     // after the last launch on each stream of the owner's
    hipStream_t stream[OWNER_STREAMS] = {};  // null: none yet
};
Turnstile g_turnstile[MAX_DEVICES];
}  // namespace

hipError_t coop_launch(const CoopOwner& who, const void* f, dim3 grid, dim3 block, void** params, unsigned lds,
                       hipStream_t st) {
    if (who.cus <= 0 || who.device < 0 || who.device >= MAX_DEVICES) return hipErrorNotSupported;
    Turnstile& t = g_turnstile[who.device];
    std::lock_guard<std::mutex> lk(t.mu);
    // (the event orders launches and publishes no data: with the system fence a
    // call of dh_propagate at N = 416 takes 4 us more, 156 against 152)
    constexpr unsigned flags = hipEventDisableTiming | hipEventDisableSystemFence;
    for (hipEvent_t& ev : t.done)
        if (!ev)
            if (hipError_t e = hipEventCreateWithFlags(&ev, flags); e != hipSuccess) return e;
    int slot = 0;
    if (t.owner == who.owner)
        while (slot < OWNER_STREAMS && t.stream[slot] && t.stream[slot] != st) ++slot;
    if (t.owner != who.owner || slot == OWNER_STREAMS) {  // another owner's turn ends
        for (int i = 0; i < OWNER_STREAMS; ++i)
            if (t.owner && t.stream[i])
                if (hipError_t e = hipEventSynchronize(t.done[i]); e != hipSuccess) return e;
        t.owner = nullptr;
        for (hipStream_t& s : t.stream) s = nullptr;
        slot = 0;
    }
    if (hipError_t e = hipLaunchCooperativeKernel(f, grid, block, params, lds, st); e != hipSuccess) return e;
    t.owner = who.owner;
    t.stream[slot] = st;
    // launched: whatever becomes of the record, the caller must not launch again
    if (hipEventRecord(t.done[slot], st) != hipSuccess) {
        (void)hipGetLastError();
        if (hipStreamSynchronize(st) != hipSuccess) (void)hipGetLastError();
        t.stream[slot] = nullptr;
    }
    return hipSuccess;
}

static std::atomic<bool> g_give_up{false};
void coop_force_give_up(bool on) { g_give_up.store(on); }
bool coop_give_up_forced() { return g_give_up.load(); }

void coop_forget(const CoopOwner& who) {
    if (who.device < 0 || who.device >= MAX_DEVICES) return;
    Turnstile& t = g_turnstile[who.device];
    std::lock_guard<std::mutex> lk(t.mu);
    if (t.owner != who.owner) return;
    t.owner = nullptr;
    for (hipStream_t& s : t.stream) s = nullptr;
}

// Work split: workgroup b owns RB = 4 RG consecutive rows; its NW waves split
// the columns (the reduction index) into NW ranges of `groups` 16-column groups.
// A group's products are FP64 MFMA 4x4x4 in 4 blocks (lanes A: 16k + 4b + i,
// B: 16k + 4b + j, D: 16i + 4b + j) with block b taking columns b, 4 + b, 8 + b,
// 12 + b of the group, so a B operand (x) feeds every row group without
// replication: lane 16k + 4b + j takes x[16g + 4k + b][j], 16 bytes (re, im).
// The ring keeps the vectors in this order (per group of 16 rows and pass of 4
// columns, the 64 lanes' values), so a load is 1 KB contiguous (as fast as
// row-major order measured, and the addresses are simpler).  A operands (H) stay
// in the lane's registers, up to what 256 registers hold beside the products (23
// groups at R = 4), and in LDS from there on.  At R = 4 a group is 8 MFMAs of 16
// cycles on one load; N = 4096: 32 groups per wave, 3.4 us of matrix-core time per
// term.
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
// All workgroups must be on the chip at once, so the launch is cooperative
// (coop_launch), and every wait is bounded (wall clock): a wave that runs out of time stops
// waiting for good, the kernel drains, and its workgroup's accumulators are
// written as NaN, which the caller's norm check turns into a repeat of the
// step with one launch per term.
//
// Copies of the flags, each polled by every RS_COPIES-th workgroup: with one
// copy the 2048 waves' polls of the same few lines queue up at one memory
// channel (a term at N = 4096, R = 4: 8.9 us with one copy, 7.6 with 8).
constexpr int RS_COPIES = 16;
constexpr unsigned long long RS_WAIT_TICKS = 200000000ull;  // 2 s of the 100 MHz wall clock
constexpr int AUX_DEVICE_SCOPE = 16;                        // buffer store: sc1

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
// z + c t with the fused operations spelt out: left to the compiler, the choice of
// the product that is fused differed between instances (NT = 32 from the others),
// and a batch member's last bits with it
__device__ __forceinline__ cplx rs_cfma(cplx c, cplx t, cplx z) {
    return cplx{fma(-c.im, t.im, fma(c.re, t.re, z.re)), fma(c.im, t.re, fma(c.re, t.im, z.im))};
}
// sum over the four blocks (lanes 4 apart of a row of 16)
__device__ __forceinline__ double rs_block_sum(double v) {
    const double z = v + rs_dpp<0x128>(v);  // row rotate 8
    return z + rs_dpp<0x124>(z);            // row rotate 4
}

// LDS contents of the workgroup are visible to all its waves past this point
// (global stores may still be in flight, unlike with __syncthreads)
__device__ __forceinline__ void rs_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// RC: column class.  1 (R <= 4): a lane's x is one complex column; 0 (R <= 2): one
// of up to 4 real columns; 2 (R <= 8): 16 real columns fill a 16x16x4 MFMA (WIDE,
// 16 rows per workgroup: A is H as loaded with lanes (k, row), B one real column
// per lane, no block sums; measured 64 cycles per 1024 products where the 4x4x4
// form takes 80 to 88), or with 8 rows (RG = 2) two sets of 4 complex columns.
// NT: the most groups per wave, a compile-time count so that the loads of x run
// ahead of the products through the whole unrolled sequence.  Groups past the
// system's own count are zero, and the order of the others (rs_first) and every
// rounding of the term are the same for each NT, so a batch member's bits do not
// depend on the larger members that share its launch (64 systems of N 256-2048, 4
// wavepackets, 40 steps: 131 to 135 ms so and with an order of its own per NT).
// blk of nblk: this workgroup's place in its system.
constexpr int rs_most(int rc) { return rc == 0 ? 24 : rc == 1 ? 23 : 22; }
constexpr int rs_max_groups(int rc) { return rc == 2 ? 30 : 32; }
// A term takes the register groups 0 .. most - 1 in order, and LDS group most + l
// after register group first + l, whose products cover its LDS reads.  first is
// that of the largest NT: with fewer LDS groups the interleaved part ends earlier,
// and a count that fits the registers has none.
constexpr int rs_first(int rc) { return 2 * rs_most(rc) - rs_max_groups(rc); }
// Groups of x in flight per wave: the loads of a term are bound by their
// latency, so as many as the registers beside H hold.  Up to 8 groups of a
// WIDE kernel this leaves room for three waves per SIMD.
constexpr int rs_depth(int rg, int nt, int nreg, int rc) {
    const int d = rg == 2    ? 6
                  : rc == 2  ? (nt > 8 ? (180 - 8 * nreg) / 8 : (88 - 8 * nreg) / 8)
                  : nreg > 20 ? 4
                             : (184 - 8 * nreg) / 4;
    return d < 2 ? std::min(2, nt) : std::min(d, nt);
}
// EAGER, while a wave's whole share of x fits its registers beside H: the data
// are their own flags.  A slot holds RS_UNSET in every word until its term is
// published; a wave loads all its groups of x at device scope (past the L2) until
// none of them is unset, which saves the wait for the stores, the flag's way and
// the second read.  A workgroup that publishes T_k sets its rows of slot k + 2
// back: every workgroup has published T_{k-1}, so all are past reading T_{k-2},
// the last term that slot may hold; and it waits for those stores before it
// publishes T_{k+1}, without which nobody looks for T_{k+2}.  Slots 0 and 1 are set
// before the launch.  A value that is itself this NaN ends in the bounded wait.
// Per term, us with flags / eager: N = 416, R = 4: 3.3 / 2.3; 1024: 3.5 / 2.6; 2048:
// 4.7 / 4.1; 2304: 4.9 / 4.5, but 2560: 5.1 / 5.7 (x no longer fits); R = 2: 2048:
// 3.7 / 2.9, 2560: 4.1 / 3.5, 3072: 4.6 / 4.4 with spills; R = 8: 1024: 4.1 / 3.3,
// 2048: 5.4 / 5.2.  A batch fills the chip, and its kernels read x past the L2
// only where that is little (640 columns).
constexpr bool rs_eager(int nw, int rg, int nt, int rc) {
    return nw == 4 ? nt <= 10 : rc == 0 ? nt <= 22 : rc == 1 ? nt <= 18 : rg == 2;
}
constexpr int RS_UNSET = 0x7ffba5c3;
__device__ __forceinline__ bool rs_unset(double x, double y) {
    return (__double2hiint(x) == RS_UNSET) | (__double2hiint(y) == RS_UNSET);
}

template <int NW, int RG, int NT, int RC>
__device__ __forceinline__ void resident_body(const ResidentArgs& a, const int blk, const int nblk) {
    constexpr bool EAGER = rs_eager(NW, RG, NT, RC);
    constexpr int NREG = RG == 4 && NT > rs_most(RC) ? rs_most(RC) : NT, NL = NT - NREG;
    constexpr int NQ = (MULTI_MAX + NW - 1) / NW;  // accumulators per wave
    constexpr bool PAIR = RC > 0, WIDE = RC == 2 && RG == 4;
    constexpr int RB = 4 * RG;
    constexpr int PT = RC == 2 && !WIDE ? 2 : 1;  // column sets
    constexpr int XL = WIDE ? 2 : PT;             // loads of x per group
    constexpr int PC = WIDE ? 8 : 4;              // columns per row of a wave's partial sums
    constexpr int DEPTH = EAGER ? NT : rs_depth(RG, NT, NREG, RC);
    using xv_t = typename std::conditional<PAIR, double2, double>::type;
    extern __shared__ double smem[];
    const int R = a.R;
    const int n = a.groups;
    double* const hs = smem;                                       // [NL][NW][RG][64]
    cplx* const part = reinterpret_cast<cplx*>(hs + NL * NW * RG * 64);  // [PT][NW][RB * PC]
    cplx* const ts = part + PT * NW * RB * PC;                           // [3][RB * R]: the last three terms' own rows
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lk = lane >> 4, lb = (lane >> 2) & 3, lj = lane & 3;
    const int N = a.N, ld = a.ld;
    const int r0 = blk * RB, k0 = w * n * 16;
    const bool active = k0 < ld;      // this wave has columns
    const int E = RB * R;             // own elements

    // H: rows r0 + 4 rg + lj, columns k0 + 16 g + 4 lk + lb (WIDE: row r0 + (lane &
    // 15), columns k0 + 16 g + 4 rg + lk, read as the transposed element: 16 lanes
    // contiguous either way); ld is a multiple of 64, so a group lies inside the
    // matrix or past it (zero) as a whole
    const int ng = active ? min(n, (ld - k0) / 16) : 0;
    double h[NREG][RG];
    const double* const hcol =
        a.H + (WIDE ? r0 + (lane & 15) + (long)ld * lk : (long)ld * (r0 + lj) + 4 * lk + lb);
    auto hval = [&](int g, int rg) {
        const long col = g < ng ? k0 + 16 * g : 0;
        const double v = hcol[WIDE ? (long)ld * (col + 4 * rg) : (long)ld * (4 * rg) + col];
        return g < ng ? v : 0.0;
    };
#pragma unroll
    for (int g = 0; g < NREG; ++g)
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) h[g][rg] = hval(g, rg);
#pragma unroll 1
    for (int g = 0; g < NL; ++g)
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) hs[((g * NW + w) * RG + rg) * 64 + lane] = hval(NREG + g, rg);

    // the wave's accumulators: q = w + NW v, elements lane + 64 u of the workgroup's rows
    constexpr int NE = (RB * (PAIR ? 4 * RC : 2) + 63) / 64;
    cplx acc[NQ][NE];
    int kq[NQ];
#pragma unroll
    for (int v = 0; v < NQ; ++v) {
        const int q = w + NW * v;
        kq[v] = q < a.m ? (a.kq ? __builtin_amdgcn_readfirstlane(a.kq[q]) : a.K) : -1;
    }
    const __amdgpu_buffer_rsrc_t ring =
        __builtin_amdgcn_make_buffer_rsrc(a.ring, 0, (int)(a.slots * a.slot_bytes), 0x00020000);
    constexpr int gbytes = XL * 64 * (int)sizeof(xv_t);  // a group's part of a slot
    // element e of the workgroup's rows goes to its lane's place (WIDE: load q
    // holds rows 8 q + k and 8 q + 4 + k of lane 16k + real column side by side)
    auto put = [&](int e, v4i bits, int slot) {
        const int row = r0 + e / R, col = e % R;
        const int to = (row >> 4) * gbytes, so = slot * a.slot_bytes;
        if constexpr (WIDE) {
            const int at = to + (row >> 3 & 1) * 1024 + (16 * (row & 3) + 2 * col) * 16 + (row >> 2 & 1) * 8;
            __builtin_amdgcn_raw_buffer_store_b64(bits.xy, ring, at, so, AUX_DEVICE_SCOPE);
            __builtin_amdgcn_raw_buffer_store_b64(bits.zw, ring, at + 16, so, AUX_DEVICE_SCOPE);
        } else {
            const int at = 16 * (row >> 2 & 3) + 4 * (row & 3) + (PAIR ? (col & 3) + 64 * (col >> 2) : 2 * col);
            __builtin_amdgcn_raw_buffer_store_b128(bits, ring, to + at * (int)sizeof(xv_t), so, AUX_DEVICE_SCOPE);
        }
    };
    auto publish = [&](int e, cplx T, int k) {  // T_k
        v4i bits;
        bits[0] = __double2loint(T.re);
        bits[1] = __double2hiint(T.re);
        bits[2] = __double2loint(T.im);
        bits[3] = __double2hiint(T.im);
        if constexpr (EAGER) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the last term's put of RS_UNSET
        put(e, bits, k % a.slots);
        if constexpr (EAGER) put(e, v4i{RS_UNSET, RS_UNSET, RS_UNSET, RS_UNSET}, (k + 2) % a.slots);
    };
    // waves 0..SW-1 add up the waves' sums and publish 64 elements each; a flag per
    // publishing wave
    constexpr int SW = RB * (PAIR ? 4 * RC : 2) > 64 ? 2 : 1;
    auto raise = [&](unsigned v) {  // after this wave's stores have arrived
        if constexpr (EAGER) return;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (lane < RS_COPIES)
            __hip_atomic_store(a.flags + (lane * nblk + blk) * SW + w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };

    // T_0 = phi (rows >= N as zero)
    if (w < SW) {
        for (int e = lane + 64 * w; e < min(E, 64 * (w + 1)); e += 64) {
            const int row = r0 + e / R;
            const cplx T = row < N ? a.phi[(long)r0 * R + e] : cplx{0.0, 0.0};
            publish(e, T, 0);
            ts[e] = T;
        }
        raise(1u);
    }
    rs_lds_barrier();
#pragma unroll
    for (int v = 0; v < NQ; ++v)
        if (kq[v] >= 0) {
            const cplx c0 = rs_coef(a.coef + (long)(w + NW * v) * a.coef_stride);
#pragma unroll
            for (int u = 0; u < NE; ++u)
                if (lane + 64 * u < E) acc[v][u] = rs_cfma(c0, ts[lane + 64 * u], cplx{0.0, 0.0});
        }

    // flags of the rows this wave reads
    const int f0 = k0 / RB, nf = active ? ((min(k0 + 16 * n, ld) + RB - 1) / RB - f0) * SW : 0;
    const unsigned* const myflag = a.flags + ((blk % RS_COPIES) * nblk + f0) * SW + min(lane, max(nf - 1, 0));
    bool dead = a.give_up != 0;
    const double a1 = 1.0 / a.r, b1 = -a.c / a.r;
    const int K = max(a.K, 1);
    for (int k = 1; k <= K; ++k) {
        cplx ck[NQ];
#pragma unroll
        for (int v = 0; v < NQ; ++v)
            if (k <= kq[v]) ck[v] = rs_coef(a.coef + (long)(w + NW * v) * a.coef_stride + k);
        if (active) {
            if (!EAGER && !dead) {
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
            if (!EAGER && slot == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            // (columns past the last are not written: their sums are not kept;
            // groups past ld read the last one: their H is zero)
            const int xoff = lane * (int)sizeof(xv_t);
            const int soff = slot * a.slot_bytes + (k0 >> 4) * gbytes;
            auto xload = [&](int g, int p) -> xv_t {
                const int so = soff + min(g, max(ng, 1) - 1) * gbytes;
                constexpr int aux = EAGER ? AUX_DEVICE_SCOPE : 0;
                if constexpr (PAIR)
                    return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(ring, xoff + p * 1024, so, aux));
                else
                    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ring, xoff, so, aux));
            };
            double yr[PT][RG], yi[PT][RG];
            v4d yw[2];  // WIDE: even and odd steps of 4 columns
#pragma unroll
            for (int p = 0; p < PT; ++p)
#pragma unroll
                for (int rg = 0; rg < RG; ++rg) yr[p][rg] = yi[p][rg] = 0.0;
            yw[0] = yw[1] = (v4d){0.0, 0.0, 0.0, 0.0};
            // the products of load p of a group with its operator values
            auto mma = [&](const double (&hv)[RG], xv_t x, int p) {
                if constexpr (WIDE) {
                    yw[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(hv[2 * p], x.x, yw[0], 0, 0, 0);
                    yw[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(hv[2 * p + 1], x.y, yw[1], 0, 0, 0);
                } else {
#pragma unroll
                    for (int rg = 0; rg < RG; ++rg) {
                        if constexpr (PAIR) {
                            yr[p][rg] = __builtin_amdgcn_mfma_f64_4x4x4f64(hv[rg], x.x, yr[p][rg], 0, 0, 0);
                            yi[p][rg] = __builtin_amdgcn_mfma_f64_4x4x4f64(hv[rg], x.y, yi[p][rg], 0, 0, 0);
                        } else {
                            yr[p][rg] = __builtin_amdgcn_mfma_f64_4x4x4f64(hv[rg], x, yr[p][rg], 0, 0, 0);
                        }
                    }
                }
            };
            constexpr int FIRST = NL > 0 ? rs_first(RC) : NT;
            auto group = [](int st) {  // of step st
                return st < FIRST ? st : st >= FIRST + 2 * NL ? st - NL
                       : (st - FIRST) % 2 == 0 ? FIRST + (st - FIRST) / 2 : NREG + (st - FIRST) / 2;
            };
            xv_t xb[DEPTH][XL];
            unsigned long long t0 = 0;
            for (int spin = 0;; ++spin) {
                if constexpr (EAGER) asm volatile("" ::: "memory");  // every look reads memory again
#pragma unroll
                for (int d = 0; d < DEPTH; ++d)
#pragma unroll
                    for (int p = 0; p < XL; ++p) xb[d][p] = xload(group(d), p);
                if (!EAGER || dead) break;
                bool unset = false;
#pragma unroll
                for (int d = 0; d < DEPTH; ++d)
#pragma unroll
                    for (int p = 0; p < XL; ++p) {
                        // columns past the last are never written
                        if constexpr (WIDE) unset |= ((lane & 15) < 2 * R) & rs_unset(xb[d][p].x, xb[d][p].y);
                        else if constexpr (PAIR) unset |= (lj + 4 * p < R) & rs_unset(xb[d][p].x, xb[d][p].y);
                        else unset |= (lj < 2 * R) & rs_unset(xb[d][p], xb[d][p]);
                    }
                if (__ballot(unset) == 0) break;
                if ((spin & 255) == 255) {
                    const unsigned long long now = wall_clock64();
                    if (t0 == 0) t0 = now;
                    else if (now - t0 > RS_WAIT_TICKS) dead = true;
                }
            }
            double hl[RG];
#pragma unroll
            for (int st = 0; st < NT; ++st) {
                const int g = group(st);
                if (st >= FIRST && st < FIRST + 2 * NL && (st - FIRST) % 2 == 0) {
#pragma unroll
                    for (int rg = 0; rg < RG; ++rg) hl[rg] = hs[(((st - FIRST) / 2 * NW + w) * RG + rg) * 64 + lane];
                }
#pragma unroll
                for (int p = 0; p < XL; ++p) {
                    const xv_t x = xb[st % DEPTH][p];
                    if (st + DEPTH < NT) xb[st % DEPTH][p] = xload(group(st + DEPTH), p);
                    if (g < NREG) mma(h[g < NREG ? g : 0], x, p);
                    else mma(hl, x, p);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (WIDE) {
                // value v of lane (k, n): row k + 4 v, real column n
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    reinterpret_cast<double*>(part)[(w * RB + lk + 4 * v) * 16 + (lane & 15)] = yw[0][v] + yw[1][v];
            } else {
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
                            part[(p * NW + w) * RB * 4 + (4 * lb + lk) * 4 + lj] = cplx{vr, vi};
                        } else if (lj < 2 * R) {  // real columns: packed as R complex ones
                            reinterpret_cast<double*>(part)[w * RB * 8 + (4 * lb + lk) * 2 * R + lj] = vr;
                        }
                    }
                }
            }
        } else {
            for (int e = lane; e < PT * RB * PC; e += 64) {
                const int p = e / (RB * PC), f = e % (RB * PC);
                part[(p * NW + w) * RB * PC + f] = cplx{0.0, 0.0};
            }
        }
        rs_lds_barrier();
        cplx* const tk = ts + (k % 3) * E;
        if (w < SW) {
            const cplx* const t1 = ts + ((k + 2) % 3) * E;
            const cplx* const t2 = ts + ((k + 1) % 3) * E;
            const double alpha = k == 1 ? a1 : 2.0 * a1, beta = k == 1 ? b1 : 2.0 * b1;
            const int e = lane + 64 * w;
            if (e < E) {
                cplx y{0.0, 0.0};
                const int row = e / R, col = e % R;
                const cplx* pp = !PAIR ? part + e : part + (WIDE ? row * 8 + col : (col / 4) * NW * RB * 4 + row * 4 + col % 4);
#pragma unroll(RG == 4 && NREG > 16 ? 4 : NW)
                for (int ww = 0; ww < NW; ++ww) {
                    y.re += pp[ww * RB * PC].re;
                    y.im += pp[ww * RB * PC].im;
                }
                const cplx xv = t1[e];
                cplx T{fma(alpha, y.re, beta * xv.re), fma(alpha, y.im, beta * xv.im)};
                if (k > 1) {
                    const cplx x2 = t2[e];
                    T.re -= x2.re;
                    T.im -= x2.im;
                }
                if (r0 + row >= N) T = cplx{0.0, 0.0};  // whatever a caller's operator has on its padded diagonal
                if (k < K) publish(e, T, k);
                tk[e] = T;
            }
            if (k < K) raise((unsigned)k + 1u);
        }
        rs_lds_barrier();
#pragma unroll
        for (int v = 0; v < NQ; ++v)
            if (k <= kq[v]) {
#pragma unroll
                for (int u = 0; u < NE; ++u)
                    if (lane + 64 * u < E) acc[v][u] = rs_cfma(ck[v], tk[lane + 64 * u], acc[v][u]);
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
    for (int v = 0; v < NQ; ++v) {
        const int q = w + NW * v;
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

template <int NW, int RG, int NT, int RC>
__global__ __launch_bounds__(NW * 64, 2) void resident_series_kernel(const ResidentArgs a) {
    resident_body<NW, RG, NT, RC>(a, blockIdx.x, gridDim.x);
}

// Several systems in one launch: workgroup i is workgroup map[i].y of member
// map[i].x (all read through the constant address space: scalar registers).
template <int NW, int NT, int RC>
__global__ __launch_bounds__(NW * 64, 2) void resident_grouped_kernel(const ResidentArgs* members, const int2* map) {
    typedef const __attribute__((address_space(4))) ResidentArgs* args_const;
    typedef const __attribute__((address_space(4))) int* int_const;
    const int_const mp = (int_const)(reinterpret_cast<const int*>(map) + 2 * blockIdx.x);
    const args_const m = (args_const)(members) + mp[0];
    ResidentArgs a;
    a.H = m->H; a.ld = m->ld; a.N = m->N; a.R = m->R; a.m = m->m; a.K = m->K; a.c = m->c; a.r = m->r;
    a.phi = m->phi; a.acc = m->acc; a.acc_stride = m->acc_stride; a.coef = m->coef; a.coef_stride = m->coef_stride;
    a.kq = m->kq; a.ring = m->ring; a.slots = m->slots; a.slot_bytes = m->slot_bytes; a.groups = m->groups;
    a.give_up = m->give_up; a.flags = m->flags;
    resident_body<NW, 4, NT, RC>(a, mp[1], a.ld / 16);
}

// Before a launch: flags to zero, and slots 0 and 1 of the ring, which lie behind
// them, to RS_UNSET.
__device__ __forceinline__ void resident_clear(const ResidentArgs& a, int first, int step) {
    const int nf = (int)(a.ring - reinterpret_cast<char*>(a.flags)) / 4, n = nf + 2 * a.slot_bytes / 4;
    for (int i = first; i < n; i += step) a.flags[i] = i < nf ? 0u : (unsigned)RS_UNSET;
}
__global__ __launch_bounds__(256) void resident_clear_kernel(ResidentArgs a) {
    resident_clear(a, blockIdx.x * 256 + threadIdx.x, gridDim.x * 256);
}
__global__ __launch_bounds__(256) void resident_clear_grouped_kernel(const ResidentArgs* members) {
    const ResidentArgs a = members[blockIdx.x];
    resident_clear(a, blockIdx.y * 256 + threadIdx.x, gridDim.y * 256);
}

// ------------------------------------------------------------------ plan
// Rows per workgroup: 16 (RG = 4), which reads x least often per product; 8 for
// R > 4 while that leaves at most 256 workgroups, twice as many CUs at work (N =
// 2048, R = 8: 5.4 against 6.6 us per term; at R = 4 8 rows measured the same as
// 16).  NT: the groups a wave needs, rounded up to even above 8 (the surplus is
// zero); for R > 4 at most 30, the rest of H no longer fits the LDS.
struct ResidentPlan {
    int RG = 0, RC = 0, NT = 0, groups = 0, wgs = 0, lds = 0;
    bool ok = false;
};

static ResidentPlan resident_plan(int ld, int R, int cus) {
    ResidentPlan p;
    if (!(R >= 1 && R <= 8) || ld <= 0 || ld > 4096) return p;
    p.RC = R <= 2 ? 0 : R <= 4 ? 1 : 2;
    p.RG = p.RC == 2 && ld <= 2048 ? 2 : 4;
    p.wgs = ld / (4 * p.RG);
    constexpr int NW = 8;
    const int n = p.groups = (ld / 16 + NW - 1) / NW;
    p.NT = n <= 8 ? n : (n + 1) / 2 * 2;
    const int np = p.RC == 2 ? 2 : 1, nl = p.RG == 4 ? std::max(0, p.NT - rs_most(p.RC)) : 0;
    p.lds = nl * NW * p.RG * 64 * 8 + np * NW * 4 * p.RG * 4 * 16 + 3 * 4 * p.RG * R * 16;
    p.ok = p.wgs <= cus && p.lds <= 160 * 1024 && (p.RC < 2 || p.NT <= 30);
    return p;
}

// bytes of one ring slot, and of the flags in front of the ring
static long resident_slot_bytes(int ld, int R) { return (long)ld * (R <= 2 ? 32 : R <= 4 ? 64 : 128); }
static long resident_flag_bytes(int ld) { return (long)RS_COPIES * (ld / 4) * 4; }
static long resident_slots(int ld, int R, long scratch_bytes) {
    const long slots = std::min(64L, (scratch_bytes - resident_flag_bytes(ld)) / resident_slot_bytes(ld, R));
    return slots < 4 ? 0 : slots;
}

bool resident_series_fits(int ld, int R, int cus, long scratch_bytes) {
    return resident_plan(ld, R, cus).ok && resident_slots(ld, R, scratch_bytes) > 0;
}

template <int RG, int NT, int RC>
static hipError_t resident_go(const ResidentArgs& a, const ResidentPlan& p, const CoopOwner& who, hipStream_t st) {
    const void* f = reinterpret_cast<const void*>(&resident_series_kernel<8, RG, NT, RC>);
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, p.lds);
    if (e != hipSuccess) return e;
    ResidentArgs arg = a;
    void* params[] = {&arg};
    return coop_launch(who, f, dim3(p.wgs), dim3(512), params, (unsigned)p.lds, st);
}

// the kernel of p.NT among LO, LO + STEP, ..., HI
template <int RG, int RC, int LO, int HI, int STEP>
static hipError_t resident_pick(const ResidentArgs& a, const ResidentPlan& p, const CoopOwner& who, hipStream_t st) {
    if (p.NT == LO) return resident_go<RG, LO, RC>(a, p, who, st);
    if constexpr (LO + STEP <= HI) return resident_pick<RG, RC, LO + STEP, HI, STEP>(a, p, who, st);
    return hipErrorInvalidValue;
}

static hipError_t resident_launch(const ResidentArgs& a, const ResidentPlan& p, const CoopOwner& who, hipStream_t st) {
    const bool few = p.NT <= 8;
    if (p.RC == 0) return few ? resident_pick<4, 0, 1, 8, 1>(a, p, who, st) : resident_pick<4, 0, 10, 32, 2>(a, p, who, st);
    if (p.RC == 1) return few ? resident_pick<4, 1, 1, 8, 1>(a, p, who, st) : resident_pick<4, 1, 10, 32, 2>(a, p, who, st);
    if (p.RG == 2) return few ? resident_pick<2, 2, 1, 8, 1>(a, p, who, st) : resident_pick<2, 2, 10, 16, 2>(a, p, who, st);
    return resident_pick<4, 2, 18, 30, 2>(a, p, who, st);
}

// scratch: flags, then as many ring slots as fit (at least 4, which the partial-sum
// buffer of a system does not hold at N <= 256 with 4 or 8 columns, nor at N <= 512
// with 6)
static bool resident_scratch(ResidentArgs* a, void* scratch, long scratch_bytes) {
    const long fb = resident_flag_bytes(a->ld), sb = resident_slot_bytes(a->ld, a->R);
    const long slots = resident_slots(a->ld, a->R, scratch_bytes);
    if (slots == 0 || a->m < 1 || a->m > MULTI_MAX) return false;
    a->flags = static_cast<unsigned*>(scratch);
    a->ring = static_cast<char*>(scratch) + fb;
    a->slots = (int)slots;
    a->slot_bytes = (int)sb;
    a->give_up = coop_give_up_forced();
    return true;
}

bool launch_resident_series(ResidentArgs a, void* scratch, long scratch_bytes, const CoopOwner& who, hipStream_t st) {
    const ResidentPlan p = resident_plan(a.ld, a.R, who.cus);
    if (!p.ok || !resident_scratch(&a, scratch, scratch_bytes)) return false;
    a.groups = p.groups;
    hipLaunchKernelGGL(resident_clear_kernel, dim3(32), dim3(256), 0, st, a);
    const hipError_t e = resident_launch(a, p, who, st);
    if (e == hipSuccess) return true;
    (void)hipGetLastError();  // not launched: the caller runs the series term by term
    return false;
}

// ------------------------------------------------------------------ batches
// A batch fills the chip with many systems, so its kernels are chosen for
// throughput: 16 rows per workgroup, both passes of R > 4 together, and 4 waves
// per workgroup as far as two such workgroups share a CU and cover each other's
// exchange (up to 256 registers a lane each and half of the LDS: ld = 2048, at
// R > 4 1920); 8 waves, one workgroup a CU, above.  The split of a system's sums
// depends on its ld and R alone: its bits are the same in every batch.  64
// systems of N 256-2048 with 4 wavepackets, 40 steps: 214 ms with one grouped
// launch per term, 153 ms with 4 waves up to ld = 1024 only, 138 up to 1408, 123
// here (1 wavepacket: 85 ms up to 1024, 63 here).
static int batch_waves(int ld, int R) { return ld <= (R > 4 ? 1920 : 2048) ? 4 : 8; }
static int batch_lds(int nw, int nt, int R) {
    const int nl = std::max(0, nt - rs_most(R <= 2 ? 0 : R <= 4 ? 1 : 2));
    return nl * nw * 4 * 64 * 8 + (R > 4 ? 2 : 1) * nw * 16 * 4 * 16 + 3 * 16 * R * 16;
}

// the grouped kernel for (waves, most groups per wave, columns), its workgroups
// per CU, and the NT it was built for
struct GroupedKernel {
    const void* f = nullptr;
    int nt = 0;
};
template <int NW, int RC>
static GroupedKernel grouped_pick(int n) {
#define DH_GROUPED(NT) \
    if (n <= NT) return GroupedKernel{reinterpret_cast<const void*>(&resident_grouped_kernel<NW, NT, RC>), NT}
    if constexpr (NW == 4) {
        DH_GROUPED(2);
        DH_GROUPED(4);
        DH_GROUPED(6);
        DH_GROUPED(8);
    }
    if constexpr (NW == 4) {
        DH_GROUPED(10);
        DH_GROUPED(12);
        DH_GROUPED(14);
    }
    DH_GROUPED(16);
    if constexpr (NW == 4) {
        DH_GROUPED(18);
        DH_GROUPED(20);
        DH_GROUPED(22);
        DH_GROUPED(24);
        DH_GROUPED(26);
        DH_GROUPED(28);
        DH_GROUPED(30);
        if constexpr (RC < 2) DH_GROUPED(32);
    }
#undef DH_GROUPED
    return GroupedKernel{};
}
static GroupedKernel grouped_kernel(int nw, int n, int R) {
    const int rc = R <= 2 ? 0 : R <= 4 ? 1 : 2;
    if (nw == 4) return rc == 0 ? grouped_pick<4, 0>(n) : rc == 1 ? grouped_pick<4, 1>(n) : grouped_pick<4, 2>(n);
    return grouped_pick<8, 2>(n);
}

bool resident_batch_member(ResidentArgs* a, void* scratch, long scratch_bytes, int cus) {
    if (cus <= 0 || a->ld > 2048 || a->R > 8 || a->ld / 16 > cus) return false;
    if (!resident_scratch(a, scratch, scratch_bytes)) return false;
    const int nw = batch_waves(a->ld, a->R);
    a->groups = (a->ld / 16 + nw - 1) / nw;
    return true;
}

// Launches: members of one wave count and about one size, as many as fit the
// chip together (largest first, so that a launch's members need about the same
// NT and take about as long).  Tried, with no gain: a member's workgroups on as
// few XCDs as hold them, different priorities or a delayed start for the
// workgroups that share a CU.
bool resident_batch_rounds(const std::vector<ResidentArgs>& members, int cus, std::vector<int2>* map,
                           std::vector<ResidentRound>* rounds) {
    map->clear();
    rounds->clear();
    std::vector<int> order(members.size());
    for (size_t i = 0; i < order.size(); ++i) order[i] = (int)i;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
        return members[x].ld != members[y].ld ? members[x].ld > members[y].ld : members[x].K > members[y].K;
    });
    int room = 0, nw = 0;
    for (int i : order) {
        const ResidentArgs& a = members[i];
        const int wgs = a.ld / 16, w = batch_waves(a.ld, a.R);
        if (w != nw || wgs > room) {
            const GroupedKernel k = grouped_kernel(w, a.groups, a.R);
            const int lds = batch_lds(w, k.nt, a.R);
            int per_cu = 0;
            if (!k.f || hipFuncSetAttribute(k.f, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess ||
                hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k.f, w * 64, (size_t)lds) != hipSuccess ||
                per_cu * cus < wgs) {
                (void)hipGetLastError();
                return false;
            }
            rounds->push_back(ResidentRound{k.f, w * 64, lds, (int)map->size(), 0});
            room = per_cu * cus;
            nw = w;
        }
        for (int g = 0; g < wgs; ++g) map->push_back(make_int2(i, g));
        rounds->back().wgs += wgs;
        room -= wgs;
    }
    return true;
}

int launch_resident_rounds(const ResidentArgs* d_members, int n, const int2* d_map,
                           const std::vector<ResidentRound>& rounds, const CoopOwner& who, hipStream_t st) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(resident_clear_grouped_kernel, dim3(n, 8), dim3(256), 0, st, d_members);
    for (const ResidentRound& r : rounds) {
        const int2* map = d_map + r.first;
        void* params[] = {&d_members, &map};
        const hipError_t e = coop_launch(who, r.f, dim3(r.wgs), dim3(r.threads), params, (unsigned)r.lds, st);
        if (e != hipSuccess) {
            set_error("resident batch series: %s", hipGetErrorString(e));
            return -1;
        }
    }
    return 0;
}

}  // namespace dh

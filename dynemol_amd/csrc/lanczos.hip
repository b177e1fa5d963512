// The Lanczos recurrence for the spectral bounds in one launch, with the operator
// resident on the chip.
//
// Step by step a recurrence of 48 steps is 48 reads of H_orth and 96 or more
// launches of a few microseconds each: 600 us at N = 514, 880 at 2078, 1440 at
// 4096.  Here a workgroup keeps its rows of H in registers (and LDS at the
// largest sizes) and every workgroup keeps the whole of v_j and v_{j-1}, spread
// over its threads.  A step exchanges one vector, y = H v_j: each workgroup
// publishes its rows of y, reads the whole of it, and forms alpha = v.y, w = y -
// alpha v - beta v_prev and beta = |w| for itself, in the same order everywhere,
// so no second exchange is needed.  The data are their own flags: every step has
// a slot of its own, set to LZ_UNSET before the launch, and a wave loads its share
// past the L2 until nothing in it is unset.  Bound by that exchange and two
// workgroup-wide sums: 126 us for the 48 steps at N = 514, 172 at 2078, 347 at
// 4096 (201, 234 and 512 with one flag per workgroup and step).
//
// All workgroups must be on the chip at once, so the launch is cooperative
// (coop_launch), and every wait is bounded (wall clock): a wave that runs out of time goes on with
// NaN, which reaches the coefficients; the caller then runs step by step.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace dh {

constexpr unsigned long long LZ_WAIT_TICKS = 200000000ull;  // 2 s of the 100 MHz wall clock
constexpr int LZ_DEVICE_SCOPE = 16;                         // buffer access: sc1
constexpr int LZ_UNSET = 0x7ffba5c3;                        // high word of a value not there yet (a NaN)

struct LanczosArgs {
    const double* H;
    int ld, N, m;
    unsigned seed;
    int give_up;  // coop_give_up_forced
    double *alpha, *beta;
    double* ring;  // y of step j at ring + j * ld
};

__device__ __forceinline__ void lz_swap32(double& a, double& b) {  // upper half of a <-> lower half of b
    const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    a = __hiloint2double(hi[0], lo[0]);
    b = __hiloint2double(hi[1], lo[1]);
}
__device__ __forceinline__ void lz_swap16(double& a, double& b) {  // odd rows of 16 of a <-> even rows of b
    const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    a = __hiloint2double(hi[0], lo[0]);
    b = __hiloint2double(hi[1], lo[1]);
}
template <int CTRL>
__device__ __forceinline__ double lz_dpp(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
// Sums of RW values over the wave: a step adds lanes 32, 16, 8, 4, 2 and 1
// apart; while more than one value is left, it also halves the values, half of
// the lanes keeping one half each.  RW = 16: 15 + 2 additions instead of 96.
// Lane l ends with the sum of value lz_row<RW>(l).
template <int RW>
__device__ __forceinline__ int lz_row(int lane) {
    if constexpr (RW == 16) return (lane >> 5 & 1) * 8 + (lane >> 4 & 1) * 4 + (lane >> 3 & 1) * 2 + (lane >> 2 & 1);
    if constexpr (RW == 8) return (lane >> 5 & 1) * 4 + (lane >> 4 & 1) * 2 + (lane >> 3 & 1);
    if constexpr (RW == 4) return (lane >> 5 & 1) * 2 + (lane >> 4 & 1);
    return lane >> 5 & 1;
}
template <int RW>
__device__ __forceinline__ double lz_wave_sums(double (&s)[RW], int lane) {
    double a[RW / 2];
#pragma unroll
    for (int i = 0; i < RW / 2; ++i) {
        lz_swap32(s[i], s[i + RW / 2]);
        a[i] = s[i] + s[i + RW / 2];
    }
    double b[RW >= 4 ? RW / 4 : 1];
    if constexpr (RW >= 4) {
#pragma unroll
        for (int i = 0; i < RW / 4; ++i) {
            lz_swap16(a[i], a[i + RW / 4]);
            b[i] = a[i] + a[i + RW / 4];
        }
    } else {
        double o = a[0];
        lz_swap16(a[0], o);
        b[0] = a[0] + o;
    }
    double c[RW >= 8 ? RW / 8 : 1];
    if constexpr (RW >= 8) {
#pragma unroll
        for (int i = 0; i < RW / 8; ++i) {
            const double keep = lane & 8 ? b[i + RW / 8] : b[i], give = lane & 8 ? b[i] : b[i + RW / 8];
            c[i] = keep + lz_dpp<0x128>(give);  // row rotate 8
        }
    } else {
        c[0] = b[0] + lz_dpp<0x128>(b[0]);
    }
    double d;
    if constexpr (RW == 16) {
        const double keep = lane & 4 ? c[1] : c[0], give = lane & 4 ? c[0] : c[1];
        d = keep + lz_dpp<0x141>(lz_dpp<0x1B>(give));  // quad reversed, then half row mirrored: 4 lanes apart
    } else {
        d = c[0] + lz_dpp<0x141>(lz_dpp<0x1B>(c[0]));
    }
    d += lz_dpp<0x4E>(d);  // quad lanes 2, 3, 0, 1
    return d + lz_dpp<0xB1>(d);  // quad lanes 1, 0, 3, 2
}

// 512 threads; wave w has columns 64 M w + 64 q + lane, q < M, of its workgroup's RW rows
template <int M>
__global__ __launch_bounds__(512) void lanczos_resident_kernel(LanczosArgs a) {
    constexpr int RW = M == 1 ? 2 : M == 2 ? 4 : M <= 4 ? 8 : 16;
    constexpr int RL = M >= 6 ? 4 : 0, RR = RW - RL;  // rows in LDS and in registers
    extern __shared__ double hs[];                    // [RL][M][512]
    __shared__ double part[8][RW], red[2][8];
    const int t = threadIdx.x, lane = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int blk = blockIdx.x, r0 = blk * RW, c0 = 64 * M * w;
    const int N = a.N, ld = a.ld;
    double h[RR][M], v[M], vp[M];
    auto hval = [&](int i, int q) {
        const int j = c0 + 64 * q + lane;
        const double x = a.H[(long)ld * (r0 + i) + min(j, ld - 1)];
        return j < ld ? x : 0.0;
    };
#pragma unroll
    for (int i = 0; i < RR; ++i)
#pragma unroll
        for (int q = 0; q < M; ++q) h[i][q] = hval(i, q);
    if constexpr (RL > 0)
        for (int i = 0; i < RL; ++i)
            for (int q = 0; q < M; ++q) hs[(i * M + q) * 512 + t] = hval(RR + i, q);
    auto block_sum = [&](double x, int buf) {
        x = wave_sum(x);
        if (lane == 0) red[buf][w] = x;
        __syncthreads();
        double s = red[buf][0];
#pragma unroll
        for (int u = 1; u < 8; ++u) s += red[buf][u];
        return s;
    };
    // the start vector of lanczos_start_kernel
    double q0 = 0.0;
#pragma unroll
    for (int q = 0; q < M; ++q) {
        const int j = c0 + 64 * q + lane;
        unsigned x = (unsigned)j * 2654435761u ^ a.seed;
        x ^= x >> 16; x *= 0x7feb352dU; x ^= x >> 15; x *= 0x846ca68bU; x ^= x >> 16;
        v[q] = j < N ? ((double)x / 4294967296.0) - 0.5 : 0.0;
        vp[q] = 0.0;
        q0 = fma(v[q], v[q], q0);
    }
    const double n0 = sqrt(block_sum(q0, 0));
#pragma unroll
    for (int q = 0; q < M; ++q) v[q] /= n0;

    const __amdgpu_buffer_rsrc_t ring =
        __builtin_amdgcn_make_buffer_rsrc(a.ring, 0, a.m * ld * 8, 0x00020000);
    bool dead = a.give_up != 0;
    double be = 0.0;
    for (int j = 0; j < a.m; ++j) {
        double s[RW];
#pragma unroll
        for (int i = 0; i < RR; ++i) {
            s[i] = 0.0;
#pragma unroll
            for (int q = 0; q < M; ++q) s[i] = fma(h[i][q], v[q], s[i]);
        }
        if constexpr (RL > 0) {
#pragma unroll
            for (int i = 0; i < RL; ++i) {
                s[RR + i] = 0.0;
#pragma unroll
                for (int q = 0; q < M; ++q) s[RR + i] = fma(hs[(i * M + q) * 512 + t], v[q], s[RR + i]);
            }
        }
        const double mine = lz_wave_sums<RW>(s, lane);
        part[w][lz_row<RW>(lane)] = mine;  // lanes of one row write the same value
        __syncthreads();
        if (w == 0) {
            if (lane < RW) {
                double y = part[0][lane];
#pragma unroll
                for (int u = 1; u < 8; ++u) y += part[u][lane];
                typedef int v2i __attribute__((ext_vector_type(2)));
                v2i bits;
                bits[0] = __double2loint(y);
                bits[1] = __double2hiint(y);
                __builtin_amdgcn_raw_buffer_store_b64(bits, ring, (j * ld + r0 + lane) * 8, 0, LZ_DEVICE_SCOPE);
            }
        }
        double y[M];
        unsigned long long t0 = 0;
        for (int spin = 0;; ++spin) {
            asm volatile("" ::: "memory");  // every look reads memory again
            bool unset = false;
#pragma unroll
            for (int q = 0; q < M; ++q) {
                const int c = c0 + 64 * q + lane;
                y[q] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ring, (j * ld + min(c, N - 1)) * 8, 0,
                                                                                       LZ_DEVICE_SCOPE));
            }
#pragma unroll
            for (int q = 0; q < M; ++q) unset |= (c0 + 64 * q + lane < N) & (__double2hiint(y[q]) == LZ_UNSET);
            if (dead || __ballot(unset) == 0) break;
            if ((spin & 255) == 255) {
                const unsigned long long now = wall_clock64();
                if (t0 == 0) t0 = now;
                else if (now - t0 > LZ_WAIT_TICKS) dead = true;
            }
        }
        double p = dead ? __builtin_nan("") : 0.0;
#pragma unroll
        for (int q = 0; q < M; ++q) {
            if (c0 + 64 * q + lane >= N) y[q] = 0.0;
            p = fma(v[q], y[q], p);
        }
        const double al = block_sum(p, 0);
        double r = 0.0;
#pragma unroll
        for (int q = 0; q < M; ++q) {
            y[q] = y[q] - al * v[q] - be * vp[q];
            r = fma(y[q], y[q], r);
        }
        const double nb = sqrt(block_sum(r, 1));
#pragma unroll
        for (int q = 0; q < M; ++q) {
            vp[q] = v[q];
            v[q] = nb > 0.0 ? y[q] / nb : 0.0;
        }
        if (nb != nb) v[0] = nb;  // a wait that ran out stays visible
        be = nb;
        if (blk == 0 && t == 0) {
            a.alpha[j] = al;
            a.beta[j + 1] = nb;
        }
    }
}

__global__ __launch_bounds__(256) void lanczos_clear_kernel(unsigned* ring, long n) {
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) ring[i] = LZ_UNSET;
}

template <int M>
static hipError_t lanczos_go(LanczosArgs a, const CoopOwner& who, hipStream_t st) {
    constexpr int RW = M == 1 ? 2 : M == 2 ? 4 : M <= 4 ? 8 : 16;
    const unsigned lds = M >= 6 ? 4 * M * 512 * 8 : 0;
    const void* f = reinterpret_cast<const void*>(&lanczos_resident_kernel<M>);
    if (hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds); e != hipSuccess) return e;
    const int wgs = (a.N + RW - 1) / RW;
    const long words = 2L * a.m * a.ld;
    hipLaunchKernelGGL(lanczos_clear_kernel, dim3((unsigned)std::min(512L, (words + 255) / 256)), dim3(256), 0, st,
                       reinterpret_cast<unsigned*>(a.ring), words);
    void* params[] = {&a};
    return coop_launch(who, f, dim3(wgs), dim3(512), params, lds, st);
}

// m steps into alpha[0..m-1], beta[1..m]; false (nothing launched that the caller
// must wait for) where the operator does not fit the chip, the device has fewer
// CUs, the scratch does not hold a vector per step, or the launch is refused
bool launch_lanczos_resident(const double* H, int ld, int N, int m, unsigned seed, double* alpha, double* beta,
                             void* scratch, long scratch_bytes, const CoopOwner& who, hipStream_t st) {
    const int M = (ld + 511) / 512, RW = M == 1 ? 2 : M == 2 ? 4 : M <= 4 ? 8 : 16;
    if (M > 8 || (N + RW - 1) / RW > who.cus) return false;
    if (8L * m * ld > scratch_bytes) return false;
    LanczosArgs a{H, ld, N, m, seed, coop_give_up_forced(), alpha, beta, static_cast<double*>(scratch)};
    hipError_t e;
    switch (M) {
        case 1: e = lanczos_go<1>(a, who, st); break;
        case 2: e = lanczos_go<2>(a, who, st); break;
        case 3: e = lanczos_go<3>(a, who, st); break;
        case 4: e = lanczos_go<4>(a, who, st); break;
        case 5: e = lanczos_go<5>(a, who, st); break;
        case 6: e = lanczos_go<6>(a, who, st); break;
        case 7: e = lanczos_go<7>(a, who, st); break;
        default: e = lanczos_go<8>(a, who, st); break;
    }
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess;
}

}  // namespace dh

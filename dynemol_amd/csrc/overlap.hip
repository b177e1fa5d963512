// STO overlap S and Wolfsberg-Helmholz Hueckel h, built on the device.
//
// The reference's two-centre scheme (overlap_D.f:144-311): for every atom pair
// (ia > ib) within the cutoff, lined-up-frame overlaps <n l m | n' l' m> (SOLAP,
// overlap_D.f:658-962) of normalised STOs (GET_ANOR, :466-517), then rotation to
// the molecular frame (ROTAR/DLMN, :983-1191).  h_ij = X_ij * S_ij
// (hamiltonians.f:33-63).
//
// The lined-up overlaps are integrated in prolate spheroidal coordinates: with
// xi in [1, inf) and eta in [-1, 1] the integrand is exp(-p xi - t eta) (p, t =
// (za +- zb) R / 2) times a polynomial of degree <= na + nb <= 10 in each, so
// 8-point Gauss-Laguerre in xi is exact and Gauss-Legendre in eta converges to
// rounding: 16 points for |t| < 4, 24 for |t| < 16, else 32 on the part of
// [-1, 1] where exp(-|t| ...) > e^-80.  The polynomial is evaluated in factored
// form (radii and heights over both centres), so nothing cancels, and a
// lane needs no tables: the recursions of the published scheme kept 7 KB of
// them per lane in scratch memory, whose traffic bound the kernel (N = 4096: 3.9
// ms; N = 514: 1.4 ms).
//
// Work decomposition: the atom pairs within the cutoff are collected into a
// list, and eight lanes take one (pair, shell pair).  A shell is the set of
// 2l+1 orbitals sharing (n, l, zeta, coef) on one atom; the lanes share the eta
// nodes of its min(la, lb) + 1 lined-up overlaps, and each writes a column of
// the (2la+1) x (2lb+1) block of S and h (and of the mirrored block).
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace dh {

// Gauss-Legendre nodes and weights, positive half: 16, 24 and 32 points
__constant__ double GL_X[36] = {
    0.09501250983763744, 0.2816035507792589, 0.45801677765722737, 0.6178762444026438, 0.755404408355003,
    0.8656312023878318, 0.9445750230732326, 0.9894009349916499,
    0.06405689286260563, 0.1911188674736163, 0.3150426796961634, 0.4337935076260451, 0.5454214713888396,
    0.6480936519369755, 0.7401241915785544, 0.820001985973903, 0.8864155270044011, 0.9382745520027328,
    0.9747285559713095, 0.9951872199970213,
    0.04830766568773832, 0.1444719615827965, 0.23928736225213706, 0.33186860228212767, 0.42135127613063533,
    0.5068999089322294, 0.5877157572407623, 0.6630442669302152, 0.7321821187402897, 0.7944837959679424,
    0.84936761373257, 0.8963211557660521, 0.9349060759377397, 0.9647622555875064, 0.9856115115452684,
    0.9972638618494816};
__constant__ double GL_W[36] = {
    0.1894506104550685, 0.18260341504492358, 0.16915651939500254, 0.14959598881657674, 0.12462897125553388,
    0.09515851168249279, 0.062253523938647894, 0.027152459411754096,
    0.12793819534675216, 0.1258374563468283, 0.12167047292780339, 0.1155056680537256, 0.10744427011596563,
    0.09761865210411388, 0.08619016153195327, 0.0733464814110803, 0.05929858491543678, 0.04427743881741981,
    0.028531388628933663, 0.0123412297999872,
    0.0965400885147278, 0.09563872007927486, 0.09384439908080457, 0.09117387869576389, 0.08765209300440381,
    0.08331192422694675, 0.07819389578707031, 0.0723457941088485, 0.06582222277636185, 0.058684093478535544,
    0.050998059262376175, 0.04283589802222668, 0.03427386291302143, 0.02539206530926206, 0.01627439473090567,
    0.007018610009470096};
// Gauss-Laguerre, 8 points
__constant__ double LAG_X[8] = {
    0.170279632305101, 0.9037017767993799, 2.2510866298661307, 4.266700170287659, 7.0459054023934655,
    10.758516010180996, 15.740678641278004, 22.863131736889265};
__constant__ double LAG_W[8] = {
    0.3691885893416375, 0.41878678081434295, 0.1757949866371718, 0.03334349226121565, 0.0027945362352256725,
    9.076508773358213e-05, 8.485746716272531e-07, 1.0480011748715104e-09};

// Lanes that share one pair of shells.  With a lane per pair of shells a small
// system leaves most of the chip idle and takes the length of one lane's
// quadrature, and a wave runs every eta tier that any of its 64 pairs needs.
// Eight lanes take the eta nodes in turn, and a column of the block each: N =
// 514: 256 -> 40 us, 2078: 415 -> 159, 4096: 692 -> 364 (three waves a SIMD; with
// four the spills cost more: 50, 203, 459).
constexpr int SUB = 8;

template <int CTRL>
__device__ __forceinline__ double ov_dpp(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double sub_sum(double v) {  // over the eight lanes, the same in each
    v += ov_dpp<0xB1>(v);         // quad lanes 1, 0, 3, 2
    v += ov_dpp<0x4E>(v);         // quad lanes 2, 3, 0, 1
    return v + ov_dpp<0x141>(v);  // the other quad of the half row
}

// Lined-up overlaps of two normalised STOs (A at the origin, B at R on z, both
// along the same axes), acc[m] += cc <n l m | n' l' m>, m = 0..min(LA, LB): the
// share of lane sub of SUB.
template <int LA, int LB>
__device__ __forceinline__ void lined_up(int na, double za, int nb, double zb, double R, double cc, int sub,
                                         double* acc) {
    constexpr int MS = LA < LB ? LA : LB;
    // Two centres at one point: the limit R -> 0 is finite, and at 1e-20 the
    // powers of 1 / p (up to the tenth) and of R still have room in the exponent
    if (R < 1e-20) R = 1e-20;
    const double hr = 0.5 * R, p = (za + zb) * hr, t = (za - zb) * hr, at = fabs(t);
    const double sg = t < 0.0 ? -1.0 : 1.0;  // exp(-t eta) is largest at eta = -sg
    const double pinv = 1.0 / p, low = fmin(za, zb) * R;  // p - |t|
    const double len = at > 40.0 ? 40.0 / at : 1.0;       // half length of the eta interval
    const int tier = at < 4.0 ? 0 : at < 16.0 ? 1 : 2;
    double sum[MS + 1];
#pragma unroll
    for (int m = 0; m <= MS; ++m) sum[m] = 0.0;
    {
        const int o = tier == 0 ? 0 : tier == 1 ? 8 : 20, half = tier == 0 ? 8 : tier == 1 ? 12 : 16;
        for (int j = sub; j < 2 * half; j += SUB) {
            const double x = j < half ? GL_X[o + j] : -GL_X[o + j - half];
            const double u = len * (1.0 + x);             // distance from the heavy end
            const double eta = sg * (u - 1.0);
            const double we = GL_W[o + (j < half ? j : j - half)] * exp(-low - at * u);
            const double e1 = 1.0 - eta * eta;
            double in[MS + 1];
#pragma unroll
            for (int m = 0; m <= MS; ++m) in[m] = 0.0;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const double xi = 1.0 + LAG_X[i] * pinv;
                const double ra = xi + eta, rb = xi - eta;          // radii, in R / 2
                const double ha = 1.0 + xi * eta, hb = xi * eta - 1.0;  // heights z_A, z_B
                const double q2 = (xi * xi - 1.0) * e1;             // distance from the axis, squared
                double f = LAG_W[i];
                for (int e = LA; e < na; ++e) f *= ra;  // r^(n-1-l) and the volume factor
                for (int e = LB; e < nb; ++e) f *= rb;
                // r^l P_l^m over rho^m of either centre
                if constexpr (LA == 1 && LB == 0) f *= ha;
                if constexpr (LA == 0 && LB == 1) f *= hb;
                if constexpr (LA == 2 && LB == 0) f *= 1.5 * ha * ha - 0.5 * ra * ra;
                if constexpr (LA == 0 && LB == 2) f *= 1.5 * hb * hb - 0.5 * rb * rb;
                if constexpr (MS == 0) {
                    in[0] += f;
                } else {
                    const double a0 = LA == 1 ? ha : 1.5 * ha * ha - 0.5 * ra * ra;
                    const double b0 = LB == 1 ? hb : 1.5 * hb * hb - 0.5 * rb * rb;
                    const double a1 = LA == 1 ? 1.0 : 3.0 * ha, b1 = LB == 1 ? 1.0 : 3.0 * hb;
                    in[0] += f * a0 * b0;
                    in[1] += f * a1 * b1 * q2;
                    if constexpr (MS == 2) in[2] += 9.0 * f * q2 * q2;
                }
            }
#pragma unroll
            for (int m = 0; m <= MS; ++m) sum[m] += we * in[m];
        }
    }
    // (R/2)^(na + nb + 1) / p, the radial norms and the norms of the harmonics
    double fa = 1.0, fb = 1.0;
    for (int i = 2; i <= 2 * na; ++i) fa *= (double)i;
    for (int i = 2; i <= 2 * nb; ++i) fb *= (double)i;
    double c = len * pinv * hr;
    const double xa = 2.0 * za * hr, xb = 2.0 * zb * hr;
    for (int i = 0; i < na; ++i) c *= xa;
    for (int i = 0; i < nb; ++i) c *= xb;
    c *= cc * 0.5 * sqrt(4.0 * za * zb * (2 * LA + 1) * (2 * LB + 1) / (fa * fb));
    // (l - m)! / (l + m)! under the root: l = 1: 1, 1/2; l = 2: 1, 1/6, 1/24
    acc[0] += c * sum[0];
    if constexpr (MS >= 1) {
        constexpr double g = LA + LB == 2 ? 0.5 : LA + LB == 3 ? 0.28867513459481288225 : 1.0 / 6.0;
        acc[1] += c * g * sum[1];
    }
    if constexpr (MS == 2) acc[2] += c * (1.0 / 24.0) * sum[2];
}

// Column m of the rotation of the real harmonics of order l (y, z, x for l = 1;
// xy, yz, z2, xz, x2-y2 for l = 2): lined-up axes e1, e2, u in the molecular frame.
// l = 2 from the traceless forms of the axes: column +-1 is (e u^T + u e^T) /
// sqrt 2, column +-2 (e1 e2^T + e2 e1^T) / sqrt 2 and (e1 e1^T - e2 e2^T) / sqrt 2.
struct Axes {
    double e1[3], e2[3], u[3];
};
__device__ __forceinline__ void d_mixed(const double* a, const double* b, double* o) {  // a, b perpendicular
    o[0] = a[0] * b[1] + a[1] * b[0];
    o[1] = a[1] * b[2] + a[2] * b[1];
    o[2] = 1.73205080756887729353 * a[2] * b[2];
    o[3] = a[0] * b[2] + a[2] * b[0];
    o[4] = a[0] * b[0] - a[1] * b[1];
}
template <int L>
__device__ __forceinline__ void rotation_column(const Axes& x, int m, double* o) {
    if constexpr (L == 0) {
        o[0] = 1.0;
    } else if constexpr (L == 1) {
        const double* v = m == 0 ? x.u : m == 1 ? x.e1 : x.e2;
        o[0] = v[1];
        o[1] = v[2];
        o[2] = v[0];
    } else if (m == 0) {
        const double* u = x.u;
        constexpr double s3 = 1.73205080756887729353;
        o[0] = s3 * u[0] * u[1];
        o[1] = s3 * u[1] * u[2];
        o[2] = 1.5 * u[2] * u[2] - 0.5;
        o[3] = s3 * u[0] * u[2];
        o[4] = 0.5 * s3 * (u[0] * u[0] - u[1] * u[1]);
    } else if (m == 1) {
        d_mixed(x.e1, x.u, o);
    } else if (m == -1) {
        d_mixed(x.e2, x.u, o);
    } else if (m == -2) {
        d_mixed(x.e1, x.e2, o);
    } else {
        const double *a = x.e1, *b = x.e2;
        o[0] = a[0] * a[1] - b[0] * b[1];
        o[1] = a[1] * a[2] - b[1] * b[2];
        o[2] = 0.86602540378443864676 * (a[2] * a[2] - b[2] * b[2]);
        o[3] = a[0] * a[2] - b[0] * b[2];
        o[4] = 0.5 * (a[0] * a[0] - b[0] * b[0] - a[1] * a[1] + b[1] * b[1]);
    }
}

// S = 0 with unit diagonal; h = 0 with h_ii = IP_i + V_shift_i.  Pad rows/cols
// in [N, ld) stay zero (the padded diagonal of S is set to one so that the
// padded Cholesky factor is the identity).
__global__ void init_SH_kernel(double* S, double* h, int N, int ld, const double* ip, const double* vshift,
                               int* count) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *count = 0;
    const long total = (long)ld * ld;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
        const int i = (int)(t % ld), j = (int)(t / ld);
        double s = 0.0, hv = 0.0;
        if (i == j) {
            s = 1.0;
            hv = i < N ? ip[i] + vshift[i] : 0.0;
        }
        S[t] = s;
        h[t] = hv;
    }
}

// Pairs (ia > ib) within the cutoff, in about basis-signature order: the lanes of
// a wave of the next kernel then share one element pair for the most part, and
// none is idle for its distance.  Atoms without orbitals have no block, and at
// most N atoms have orbitals, so the list holds at most N (N - 1) / 2 pairs
// whatever n_atoms is.
__global__ __launch_bounds__(256) void pair_list_kernel(const BasisDev b, double cutoff, int* count, int2* list) {
    const long npair = (long)b.n_atoms * (b.n_atoms - 1) / 2;
    const long q = blockIdx.x * 256L + threadIdx.x;
    int2 pr = make_int2(0, 0);
    bool near = false;
    if (q < npair) {
        // q -> (p > r): q = p*(p-1)/2 + r
        int p = (int)((1.0 + sqrt(1.0 + 8.0 * (double)q)) * 0.5);
        while ((long)p * (p - 1) / 2 > q) --p;
        while ((long)(p + 1) * p / 2 <= q) ++p;
        const int r = (int)(q - (long)p * (p - 1) / 2);
        const int ap = b.atom_order[p], ar = b.atom_order[r];
        const double x = b.coords[3 * ap] - b.coords[3 * ar], y = b.coords[3 * ap + 1] - b.coords[3 * ar + 1],
                     z = b.coords[3 * ap + 2] - b.coords[3 * ar + 2];
        near = b.atom_nshell[ap] > 0 && b.atom_nshell[ar] > 0 && !(sqrt(x * x + y * y + z * z) > cutoff);
        pr = make_int2(ap, ar);
    }
    const unsigned long long mask = __ballot(near);
    const int lane = threadIdx.x & 63;
    int base = 0;
    if (lane == 0 && mask) base = atomicAdd(count, __popcll(mask));
    base = __shfl(base, 0);
    if (near) list[base + __popcll(mask & ((1ull << lane) - 1))] = pr;
}

template <int LA, int LB>
__device__ __forceinline__ void shell_block(const BasisDev& b, int shA, int shB, const Axes& ax, double R, double* S,
                                            double* h, int ld, double s_drop, int sub) {
    constexpr int MS = LA < LB ? LA : LB;
    double sig[MS + 1];
#pragma unroll
    for (int m = 0; m <= MS; ++m) sig[m] = 0.0;
    for (int j = 0; j < b.sh_nzeta[shB]; ++j)
        for (int i = 0; i < b.sh_nzeta[shA]; ++i)
            lined_up<LA, LB>(b.sh_n[shA], b.sh_zeta[2 * shA + i], b.sh_n[shB], b.sh_zeta[2 * shB + j], R,
                             b.sh_coef[2 * shA + i] * b.sh_coef[2 * shB + j], sub, sig);
#pragma unroll
    for (int m = 0; m <= MS; ++m) sig[m] = sub_sum(sig[m]);
    double col[2 * LA + 1];  // column sub of the block (lanes past its last repeat it and store nothing)
#pragma unroll
    for (int m = -MS; m <= MS; ++m) {
        double ra[2 * LA + 1], rb[2 * LB + 1];
        rotation_column<LA>(ax, m, ra);
        rotation_column<LB>(ax, m, rb);
        double sb = rb[0];
#pragma unroll
        for (int j = 1; j <= 2 * LB; ++j) sb = sub == j ? rb[j] : sb;
        const double s = sig[m < 0 ? -m : m];
#pragma unroll
        for (int i = 0; i <= 2 * LA; ++i) {
            const double v = s * ra[i] * sb;
            col[i] = m == -MS ? v : col[i] + v;
        }
    }
    if (sub > 2 * LB) return;
    const int a0 = b.sh_orb0[shA], bo = b.sh_orb0[shB] + sub;
    // X of the block: IP, k_WH and V_shift per orbital
#pragma unroll
    for (int i = 0; i <= 2 * LA; ++i) {
        double s = col[i];
        if (fabs(s) < s_drop) s = 0.0;
        const int a = a0 + i;
        const double hv = huckel_x(b.ip[a], b.ip[bo], b.kwh[a], b.kwh[bo], b.vshift[a], b.vshift[bo]) * s;
        S[(long)a + (long)ld * bo] = s;
        S[(long)bo + (long)ld * a] = s;
        h[(long)a + (long)ld * bo] = hv;
        h[(long)bo + (long)ld * a] = hv;
    }
}

__global__ __launch_bounds__(64, 3) void build_SH_kernel(const BasisDev b, const int* count, const int2* list, double* S,
                                                      double* h, int ld, double s_drop) {
    const int q = blockIdx.x * (64 / SUB) + threadIdx.x / SUB, sub = threadIdx.x % SUB;
    if (q >= *count) return;
    const int2 pr = list[q];
    const int sp = blockIdx.y;
    // the reference's roles: A is the atom of higher index (overlap_D.f:144-311)
    const bool p_is_a = pr.x > pr.y;
    const int ia = p_is_a ? pr.x : pr.y, ib = p_is_a ? pr.y : pr.x;
    const int sa = p_is_a ? sp / MAX_SHELLS : sp % MAX_SHELLS;
    const int sb = p_is_a ? sp % MAX_SHELLS : sp / MAX_SHELLS;
    if (sa >= b.atom_nshell[ia] || sb >= b.atom_nshell[ib]) return;
    Axes ax;
    double R = 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        ax.u[d] = b.coords[3 * ib + d] - b.coords[3 * ia + d];
        R += ax.u[d] * ax.u[d];
    }
    R = sqrt(R);
#pragma unroll
    for (int d = 0; d < 3; ++d) ax.u[d] /= R;
    // e1 = axis x u for the coordinate axis farthest from u, e2 = u x e1
    const double ux = fabs(ax.u[0]), uy = fabs(ax.u[1]), uz = fabs(ax.u[2]);
    if (ux <= uy && ux <= uz) {
        ax.e1[0] = 0.0; ax.e1[1] = -ax.u[2]; ax.e1[2] = ax.u[1];
    } else if (uy <= uz) {
        ax.e1[0] = ax.u[2]; ax.e1[1] = 0.0; ax.e1[2] = -ax.u[0];
    } else {
        ax.e1[0] = -ax.u[1]; ax.e1[1] = ax.u[0]; ax.e1[2] = 0.0;
    }
    const double n1 = 1.0 / sqrt(ax.e1[0] * ax.e1[0] + ax.e1[1] * ax.e1[1] + ax.e1[2] * ax.e1[2]);
#pragma unroll
    for (int d = 0; d < 3; ++d) ax.e1[d] *= n1;
    ax.e2[0] = ax.u[1] * ax.e1[2] - ax.u[2] * ax.e1[1];
    ax.e2[1] = ax.u[2] * ax.e1[0] - ax.u[0] * ax.e1[2];
    ax.e2[2] = ax.u[0] * ax.e1[1] - ax.u[1] * ax.e1[0];
    const int shA = b.atom_shell0[ia] + sa, shB = b.atom_shell0[ib] + sb;
    switch (3 * b.sh_l[shA] + b.sh_l[shB]) {
        case 0: shell_block<0, 0>(b, shA, shB, ax, R, S, h, ld, s_drop, sub); break;
        case 1: shell_block<0, 1>(b, shA, shB, ax, R, S, h, ld, s_drop, sub); break;
        case 2: shell_block<0, 2>(b, shA, shB, ax, R, S, h, ld, s_drop, sub); break;
        case 3: shell_block<1, 0>(b, shA, shB, ax, R, S, h, ld, s_drop, sub); break;
        case 4: shell_block<1, 1>(b, shA, shB, ax, R, S, h, ld, s_drop, sub); break;
        case 5: shell_block<1, 2>(b, shA, shB, ax, R, S, h, ld, s_drop, sub); break;
        case 6: shell_block<2, 0>(b, shA, shB, ax, R, S, h, ld, s_drop, sub); break;
        case 7: shell_block<2, 1>(b, shA, shB, ax, R, S, h, ld, s_drop, sub); break;
        default: shell_block<2, 2>(b, shA, shB, ax, R, S, h, ld, s_drop, sub); break;
    }
}

// scratch: a counter, then up to N (N - 1) / 2 pairs (8 bytes each)
int launch_build_SH(const BasisDev& b, int N, int ld, double* S, double* h, double cutoff, double s_drop, void* scratch,
                    hipStream_t st) {
    int* const count = static_cast<int*>(scratch);
    int2* const list = reinterpret_cast<int2*>(static_cast<char*>(scratch) + 256);
    {
        const long total = (long)ld * ld;
        int blocks = (int)std::min<long>((total + 255) / 256, 8192);
        hipLaunchKernelGGL(init_SH_kernel, dim3(blocks), dim3(256), 0, st, S, h, N, ld, b.ip, b.vshift, count);
    }
    const long npair = (long)b.n_atoms * (b.n_atoms - 1) / 2;
    if (npair > 0) {
        hipLaunchKernelGGL(pair_list_kernel, dim3((unsigned)((npair + 255) / 256)), dim3(256), 0, st, b, cutoff, count,
                           list);
        hipLaunchKernelGGL(build_SH_kernel, dim3((unsigned)((npair + 64 / SUB - 1) / (64 / SUB)), MAX_SHELLS * MAX_SHELLS), dim3(64), 0, st,
                           b, count, list, S, h, ld, s_drop);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace dh

// kernels_init.hip -- IP-Glasma initial conditions on the device.
//
//   k_tp          T_p sums over nucleons            (Init.cpp:1009-1115)
//   k_qs_b/_a     Q_s^2(T_p, y) fixed point -> g^2mu^2 (Init.cpp:1219-1421)
//   k_qs_serial   the same loop in the reference's single-thread site order,
//                 used when a site would read the previous site's Q_s
//   k_stats       <Q_s>, T_pp and the success test inputs (Init.cpp:1423-1618)
//   k_setv_*      rho = g sqrt(g2mu2/Ny) z, 2D FFT, 1/(k^2+m^2) e^{-|k|UVdamp},
//                 inverse FFT, V <- exp(-i A.t) V  (Init.cpp:1678-1850)
//   k_links       U^(1,2)_{x,y} = V(x) V(x+i)^+ with the NaN guard
//                 (Init.cpp:2459-2491)
//   k_newton_quad, k_newton, k_newton_polish  per-link root finder
//                 (Init.cpp:3344-3481)
//   k_pi_init     pi = -(2i/g) A^eta (Init.cpp:2521-2584, 2664-2680)
#include <algorithm>

#include "ipg_device.hpp"
#include "ipg_internal.hpp"
#include "fft_lds.hpp"
#include "solve_rows.hpp"
#include "adjoint.hpp"

namespace {

constexpr double HBARC = 0.1973269718;  // Phys_consts.h:6

// ---- Philox4x32-10 and the colour-charge counter map -------------------------
__device__ __forceinline__ void philox(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; r++) {
        if (r > 0) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        // one 64-bit product (v_mad_u64_u32) instead of a high and a low one:
        // integer multiplies take four times the issue slots of an add
        const uint64_t m0 = (uint64_t)0xD2511F53u * c[0], m1 = (uint64_t)0xCD9E8D57u * c[2];
        const uint32_t hi0 = (uint32_t)(m0 >> 32), lo0 = (uint32_t)m0;
        const uint32_t hi1 = (uint32_t)(m1 >> 32), lo1 = (uint32_t)m1;
        uint32_t n0 = hi1 ^ c[1] ^ k0, n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0;
        c[1] = lo1;
        c[2] = n2;
        c[3] = lo0;
    }
}
__device__ __forceinline__ double u53(uint32_t lo, uint32_t hi) {
    uint64_t x = ((uint64_t)hi << 32) | lo;
    return ((double)(x >> 11) + 0.5) * (1.0 / 9007199254740992.0);
}
// counter {site, slice k, nucleus/tag, pair p}, key = seed; Box-Muller
__device__ __forceinline__ void normals8(uint64_t seed, uint32_t c1, uint32_t c2, uint32_t s, double z[8]) {
#pragma unroll
    for (uint32_t p = 0; p < 4; p++) {
        uint32_t c[4] = {s, c1, c2, p};
        philox(c, (uint32_t)seed, (uint32_t)(seed >> 32));
        double r = sqrt(-2.0 * log(u53(c[0], c[1])));
        // sin and cos of 2 pi u2 as sincospi(2 u2): the doubling is exact,
        // the reduction of the argument cheaper than sincos's (the oracle's
        // cos(2 pi u2) differs by the rounding of 2 pi u2, ~1e-16)
        double sn, cs;
        sincospi(2.0 * u53(c[2], c[3]), &sn, &cs);
        z[2 * p] = r * cs;
        z[2 * p + 1] = r * sn;
    }
}

// ---- T_p -----------------------------------------------------------------------
// A nucleon's thickness is a Gaussian in the distance b to it; without the
// proton anisotropy (xi = 0) it factorises over the lattice axes,
// exp(-b^2 / (2 BG hbarc^2)) = gx(n, i) gy(n, j), so k_tp_g tabulates the
// 2 (A1 + A2) N factors (one exp per nucleon and lattice line, in the
// transform buffer, which setV has not yet taken) and k_tp sums their
// products: one multiply per nucleon and site instead of one exp.  With
// xi != 0, or a table that would not fit, k_tp takes the exp per nucleon and
// site (the reference's own order, Init.cpp:1009-1115).
__device__ __forceinline__ bool tp_separable(const EvDesc& ev) {
    return ev.xi == 0. && 2LL * (ev.A1 + ev.A2) * ev.N <= 72LL * (long long)ev.S;
}
__global__ __launch_bounds__(IPG_BLOCK) void k_tp_g(const EvDesc* __restrict__ evs, int nev) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active || !tp_separable(ev)) return;
    const int A = ev.A1 + ev.A2, N = ev.N;
    const long long AN = (long long)A * N, stride = (long long)ev.nblocks * IPG_BLOCK;
    double* g = reinterpret_cast<double*>(ev.fftbuf);  // [gx: A][N], then [gy: A][N]
    for (long long t = (long long)(blockIdx.x - ev.block0) * IPG_BLOCK + threadIdx.x; t < 2 * AN; t += stride) {
        const int xy = t >= AN;
        const long long r = t - xy * AN;
        const int n = (int)(r / N), i = (int)(r - (long long)n * N);
        const double d = ev.nuc[4 * n + xy] - (-ev.L / 2. + ev.a * i);
        g[t] = exp(-(d * d / (HBARC * HBARC)) / (2. * ev.BG));
    }
}
// N a multiple of 64: a block takes 4 rows x 64 columns; each wavefront sums
// one nucleus for two of the rows, a column a lane, so a load of gy serves two
// products and gx is uniform (a thread per site loads both factors for every
// product: 125 us at N = 512 with 416 nucleons, 57 us at N = 128; this
// 56 and 17 us).  The nucleons are summed one after the other as in the
// other path, so the two agree to the last bit; quarters of the list summed
// apart would be faster by a few microseconds and round differently.  Other
// N: a thread per site.
__global__ __launch_bounds__(IPG_BLOCK) void k_tp(const EvDesc* __restrict__ evs, int nev) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active) return;
    const int N = ev.N;
    const int lb = xcd_remap(blockIdx.x - ev.block0, ev.nblocks);
    if ((N & 63) == 0 && tp_separable(ev)) {
        if ((long long)lb * IPG_BLOCK >= ev.S) return;
        const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63);
        const int cpr = N >> 6, i0 = 4 * (lb / cpr) + 2 * (w >> 1), j0 = 64 * (lb % cpr);
        const int A = ev.A1 + ev.A2, n1 = w & 1 ? A : ev.A1;
        const double* gx = reinterpret_cast<const double*>(ev.fftbuf) + i0;
        const double* gy = reinterpret_cast<const double*>(ev.fftbuf) + (size_t)A * N + j0 + lane;
        double t0 = 0., t1 = 0.;
#pragma unroll 16
        for (int n = w & 1 ? ev.A1 : 0; n < n1; n++) {
            const double y = gy[(size_t)n * N];
            t0 += gx[(size_t)n * N] * y;
            t1 += gx[(size_t)n * N + 1] * y;
        }
        double* o = (w & 1 ? ev.TpB : ev.TpA) + (size_t)i0 * N + j0 + lane;
        const double pre = sqrt(1 + ev.xi), nrm = 2. * M_PI * ev.BG;
        o[0] = pre * t0 / nrm;
        o[N] = pre * t1 / nrm;
        return;
    }
    const long long s = (long long)lb * IPG_BLOCK + threadIdx.x;
    if (s >= ev.S) return;
    const int ix = (int)(s / N), iy = (int)(s - (long long)ix * N);
    const double xi = ev.xi, BG = ev.BG;
    const double pre = sqrt(1 + xi), nrm = 2. * M_PI * BG;
    double tA = 0., tB = 0.;
    if (tp_separable(ev)) {
        const int A = ev.A1 + ev.A2;
        const double* gx = reinterpret_cast<const double*>(ev.fftbuf) + ix;
        const double* gy = reinterpret_cast<const double*>(ev.fftbuf) + (size_t)A * N + iy;
        for (int n = 0; n < ev.A1; n++) tA += gx[(size_t)n * N] * gy[(size_t)n * N];
        for (int n = ev.A1; n < A; n++) tB += gx[(size_t)n * N] * gy[(size_t)n * N];
        ev.TpA[s] = pre * tA / nrm;
        ev.TpB[s] = pre * tB / nrm;
        return;
    }
    const double x = -ev.L / 2. + ev.a * ix, y = -ev.L / 2. + ev.a * iy;
    for (int n = 0; n < ev.A1 + ev.A2; n++) {
        const double xm = ev.nuc[4 * n], ym = ev.nuc[4 * n + 1];
        double dx = xm - x, dy = ym - y;
        double bp2 = dx * dx + dy * dy;
        // the anisotropy term xi (b.n)^2 is exactly +0 for xi = 0
        if (xi != 0.) {
            const double ph = ev.nuc[4 * n + 2];
            const double pr = dx * cos(ph) + dy * sin(ph);
            bp2 = bp2 + xi * (pr * pr);
        }
        bp2 /= HBARC * HBARC;
        double T = pre * exp(-bp2 / (2. * BG)) / nrm;
        if (n < ev.A1)
            tA = tA + T;
        else
            tB = tB + T;
    }
    ev.TpA[s] = tA;
    ev.TpB[s] = tB;
}

// ---- Q_s^2 -------------------------------------------------------------------------
constexpr int NT = 200, NYQ = 44;

// getNuclearQs2 (Init.cpp:686-749); the interval search is a bisection, which
// finds the same unique interval of the increasing T list as the linear scan
__device__ double nuclear_qs2(const double* __restrict__ Tl, const double* __restrict__ Q, double T, double y) {
    const double dy = 0.25;
    const int posy = (int)floor(y / dy + 0.0000001);
    const int tot = NT * NYQ;
    auto q = [&](int it, int iy) {
        int k = it * NYQ + iy;
        return Q[k < tot ? k : tot - 1];
    };
    if (y > NYQ * dy) return NAN;
    if (T > Tl[NT - 1]) {
        double fy = (y - (double)posy * dy) / dy;
        return fy * q(NT - 1, posy + 1) + (1. - fy) * q(NT - 1, posy);
    }
    if (T < Tl[0]) return 0.;
    if (!(T >= Tl[0] && T < Tl[NT - 1])) {
        // NaN or T equal to the last node: the reference's fallback
        double fy = T == Tl[NT - 1] ? (y - (double)posy * dy) / dy : 0.;
        return fy * q(NT - 1, posy + 1) + (1. - fy) * q(NT - 1, posy);
    }
    int lo = 0, hi = NT - 1;  // Tl[lo] <= T < Tl[hi]
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (T >= Tl[mid])
            lo = mid;
        else
            hi = mid;
    }
    double fT = (T - Tl[lo]) / (Tl[lo + 1] - Tl[lo]);
    double fy = (y - (double)posy * dy) / dy;
    double dn = fT * q(lo + 1, posy) + (1. - fT) * q(lo, posy);
    double up = fT * q(lo + 1, posy + 1) + (1. - fT) * q(lo, posy + 1);
    return fy * up + (1. - fy) * dn;
}

__device__ __forceinline__ double distance_of(double BG, double Tp, double rmax) {
    double l = log(2 * M_PI * BG * Tp);
    if (l < 0.) {
        if (isinf(l)) return rmax + 1.;
        return sqrt(-2. * BG * l) * HBARC;
    }
    return 0.;
}

// one fixed-point run for one nucleus; ly and Qs carry in and out
__device__ double qs_fixed_point(const double* Tl, const double* Q, double Tp, double& ly, double& Qs,
                                 double yIn, double sgn, double ratio, const EvDesc& ev) {
    const double expo = 5.6;
    double g2 = 0.;
    double ydev = 10000;
    const double ey = exp(sgn * yIn);
    // the reference loops without bound; a cap keeps every wave finite
    for (int guard = 0; fabs(ydev) > 0.001 && guard < 100000; guard++) {
        if (ly >= 0) {
            Qs = sqrt(nuclear_qs2(Tl, Q, Tp, fabs(ly)));
        } else {
            double xv = Qs * ev.xFactor / ev.roots * ey;
            if (xv == 0)
                Qs = 0.;
            else
                Qs = sqrt(nuclear_qs2(Tl, Q, Tp, 0.)) * sqrt(pow((1 - xv) / (1 - 0.01), expo) * pow((0.01 / xv), 0.2));
        }
        if (Qs == 0) {
            ydev = 0;
            g2 = 0.;
        } else {
            g2 = Qs * Qs / ratio / ratio * ev.a * ev.a / HBARC / HBARC / ev.g / ev.g;
            double ynew = log(0.01 / (Qs * ev.xFactor / ev.roots * ey));
            ydev = ly - ynew;
            ly = ynew;
        }
    }
    if (g2 != g2) g2 = 0.;
    return g2;
}

__device__ __forceinline__ int site_check2(const EvDesc& ev, long long s) {
    double dA = distance_of(ev.BG, ev.TpA[s], ev.rmax);
    double dB = distance_of(ev.BG, ev.TpB[s], ev.rmax);
    int check = 0;
    if (dA < ev.rmax) check = 1;
    if (dB < ev.rmax && check == 1) check = 2;
    return check == 2;
}

// block maximum of an int (all threads of the block call it), valid in thread 0
__device__ int block_max_int(int v) {
    __shared__ int w[IPG_BLOCK / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_down(v, o, 64));
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
    __syncthreads();
    int r = -1;
    if (threadIdx.x == 0)
        for (int k = 0; k < IPG_BLOCK / 64; k++) r = max(r, w[k]);
    __syncthreads();
    return r;
}

// partial slot holding, per block, the last site whose check2 flag is set
constexpr int kSlotCheck2 = 8;

// pass 1: nucleus B from the input rapidity at every site; records per block
// the last site inside both nuclei (for the site order of pass 2)
__global__ __launch_bounds__(IPG_BLOCK) void k_qs_b(const EvDesc* __restrict__ evs, int nev, const double* Tl,
                                                   const double* Q, int* flag) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (blockIdx.x == (unsigned)ev.block0 && threadIdx.x == 0) flag[e] = 0;
    if (!ev.active) return;
    const int lb = xcd_remap(blockIdx.x - ev.block0, ev.nblocks);
    const long long s = (long long)lb * IPG_BLOCK + threadIdx.x;
    int c2 = 0;
    if (s < ev.S) {
        c2 = site_check2(ev, s);
        ev.check2[s] = c2;
        ev.g2A[s] = 0.;
        ev.g2B[s] = 0.;
        ev.yB[s] = ev.rapidity;
        if (c2 && ev.useFluctuatingx == 1) {
            double ly = ev.rapidity, Qs = 1.;
            ev.g2B[s] = qs_fixed_point(Tl, Q, ev.TpB[s], ly, Qs, ev.rapidity, -1., ev.QsmuRatioB, ev);
            ev.yB[s] = ly;
        }
    }
    const int last = block_max_int(c2 ? (int)s : -1);
    if (threadIdx.x == 0) ev.partial[(size_t)kSlotCheck2 * ev.nblocks + lb] = (double)last;
}

// the last site before s inside both nuclei (-1: none): a walk back through
// s's own block, then through the per-block maxima of earlier blocks
__device__ long long prev_check2(const EvDesc& ev, long long s) {
    const long long b0 = (s / IPG_BLOCK) * IPG_BLOCK;
    for (long long q = s - 1; q >= b0; q--)
        if (ev.check2[q]) return q;
    for (long long b = s / IPG_BLOCK - 1; b >= 0; b--) {
        const double m = ev.partial[(size_t)kSlotCheck2 * ev.nblocks + b];
        if (m >= 0.) return (long long)m;
    }
    return -1;
}

// pass 2: nucleus A starting from the previous check2 site's final B rapidity
__global__ __launch_bounds__(IPG_BLOCK) void k_qs_a(const EvDesc* __restrict__ evs, int nev, const double* Tl,
                                                   const double* Q, int* flag) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active) return;
    const long long s = (long long)xcd_remap(blockIdx.x - ev.block0, ev.nblocks) * IPG_BLOCK + threadIdx.x;
    if (s >= ev.S) return;
    if (!ev.check2[s]) return;
    if (ev.useFluctuatingx == 1) {
        const long long p = prev_check2(ev, s);
        double ly = p >= 0 ? ev.yB[p] : ev.rapidity;
        if (ly < 0 || ev.rapidity < 0) {
            // the first iteration would read Q_s carried from the previous site
            atomicOr(&flag[e], 1);
            return;
        }
        double Qs = 1.;
        ev.g2A[s] = qs_fixed_point(Tl, Q, ev.TpA[s], ly, Qs, ev.rapidity, 1., ev.QsmuRatio, ev);
    } else {
        // fixed x: Q_s^2 at the input rapidity (Init.cpp:1393-1406)
        double y = ev.rapidity;
        ev.g2A[s] = nuclear_qs2(Tl, Q, ev.TpA[s], y) / ev.QsmuRatio / ev.QsmuRatio * ev.a * ev.a / HBARC / HBARC /
                    ev.g / ev.g;
        ev.g2B[s] = nuclear_qs2(Tl, Q, ev.TpB[s], y) / ev.QsmuRatioB / ev.QsmuRatioB * ev.a * ev.a / HBARC /
                    HBARC / ev.g / ev.g;
    }
}

// the reference's single-thread loop, one thread per event (rare fallback)
__global__ void k_qs_serial(const EvDesc* __restrict__ evs, int nev, const double* Tl, const double* Q,
                            const int* flag) {
    const int e = blockIdx.x;
    if (e >= nev || threadIdx.x != 0) return;
    const EvDesc& ev = evs[e];
    if (!ev.active || !(flag[e] & 1)) return;
    double ly = ev.rapidity, QsA = 1., QsB = 1.;
    for (long long s = 0; s < ev.S; s++) {
        ev.g2A[s] = 0.;
        ev.g2B[s] = 0.;
        if (!ev.check2[s]) continue;
        ev.g2A[s] = qs_fixed_point(Tl, Q, ev.TpA[s], ly, QsA, ev.rapidity, 1., ev.QsmuRatio, ev);
        ly = ev.rapidity;
        ev.g2B[s] = qs_fixed_point(Tl, Q, ev.TpB[s], ly, QsB, ev.rapidity, -1., ev.QsmuRatioB, ev);
    }
}

// ---- statistics (Init.cpp:1423-1518) ---------------------------------------------
__device__ __forceinline__ double wsum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}

constexpr int kNearCap = 512;
// out per block: 7 partial sums (aQs, aQs2, aQs2Avg, aQs2min, aQs2min2, count, Tpp)
__global__ __launch_bounds__(IPG_BLOCK) void k_stats(const EvDesc* __restrict__ evs, int nev) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active) return;
    const int lb = xcd_remap(blockIdx.x - ev.block0, ev.nblocks);
    const long long s = (long long)lb * IPG_BLOCK + threadIdx.x;
    // the wounded nucleons within rcut of the block's sites (a superset, by the
    // rows and, inside one row, the columns it covers); the loop over all of
    // them per site was 130 us of the kernel's 146 at N = 512 with 416
    // nucleons.  A list that would not fit falls back to that loop.
    __shared__ int near_idx[2][kNearCap];
    __shared__ int near_n[2];
    if (threadIdx.x < 2) near_n[threadIdx.x] = 0;
    __syncthreads();
    {
        const int N = ev.N;
        const int b0 = lb * IPG_BLOCK, b1 = b0 + IPG_BLOCK - 1;
        const int r0 = b0 / N, r1 = b1 / N;
        const double x0 = -ev.L / 2. + ev.a * r0, x1 = -ev.L / 2. + ev.a * r1;
        const double y0 = r0 == r1 ? -ev.L / 2. + ev.a * (b0 - r0 * N) : -ev.L / 2.;
        const double y1 = r0 == r1 ? -ev.L / 2. + ev.a * (b1 - r0 * N) : ev.L / 2.;
        const double reach = ev.rcut * (1. + 1e-6);
        for (int n = threadIdx.x; n < ev.A1 + ev.A2; n += IPG_BLOCK) {
            const double px = ev.nuc[4 * n], py = ev.nuc[4 * n + 1];
            if (ev.nuc[4 * n + 3] == 1. && px > x0 - reach && px < x1 + reach && py > y0 - reach && py < y1 + reach) {
                const int nb = n >= ev.A1;
                const int q = atomicAdd(&near_n[nb], 1);
                if (q < kNearCap) near_idx[nb][q] = n;
            }
        }
    }
    __syncthreads();
    double v[7] = {0, 0, 0, 0, 0, 0, 0};
    if (s < ev.S) {
        const int N = ev.N;
        const int ix = (int)(s / N), iy = (int)(s - (long long)ix * N);
        const double x = -ev.L / 2. + ev.a * ix, y = -ev.L / 2. + ev.a * iy;
        const double rcut = ev.rcut;
        const double a = ev.a, g = ev.g, rA = ev.QsmuRatio, rB = ev.QsmuRatioB;
        const double g2A = (s > 0 && s < (long long)(N - 1) * N + N - 1) ? ev.g2A[s] : 0.;
        const double g2B = (s > 0 && s < (long long)(N - 1) * N + N - 1) ? ev.g2B[s] : 0.;
        const double fA = rA * rA / a / a * HBARC * HBARC * g * g, fB = rB * rB / a / a * HBARC * HBARC * g * g;
        v[4] = g2B >= g2A ? g2A * fA : g2B * fB;
        // a wounded nucleon of A, then one of B, within rcut; the squared
        // distance decides away from rcut^2 (margins of 1e-12 keep every
        // such decision equal to sqrt(d^2) < rcut), sqrt only next to it
        const double in2 = rcut * rcut * (1. - 1e-12), out2 = rcut * rcut * (1. + 1e-12);
        auto near = [&](int n) {
            const double dx = x - ev.nuc[4 * n], dy = y - ev.nuc[4 * n + 1];
            const double d2 = dx * dx + dy * dy;
            const bool inside = d2 < in2 || (d2 <= out2 && sqrt(d2) < rcut);
            return inside && ev.nuc[4 * n + 3] == 1.;
        };
        int check = 0;
        if (near_n[0] <= kNearCap && near_n[1] <= kNearCap) {
            for (int q = 0; q < near_n[0] && check == 0; q++)
                if (near(near_idx[0][q])) check = 1;
            if (check == 1)
                for (int q = 0; q < near_n[1] && check == 1; q++)
                    if (near(near_idx[1][q])) check = 2;
        } else {
            for (int n = 0; n < ev.A1 && check == 0; n++)
                if (near(n)) check = 1;
            if (check == 1)
                for (int n = ev.A1; n < ev.A1 + ev.A2 && check == 1; n++)
                    if (near(n)) check = 2;
        }
        if (check == 2) {
            if (g2B > g2A) {
                v[0] = sqrt(g2B * fB);
                v[1] = g2B * fB;
                v[3] = g2A * fA;
            } else {
                v[0] = sqrt(g2A * fA);
                v[1] = g2A * fA;
                v[3] = g2B * fB;
            }
            v[2] = (g2B * rB * rB + g2A * rA * rA) / 2. / a / a * HBARC * HBARC * g * g;
            v[5] = 1.;
        }
        v[6] = ev.TpB[s] * ev.TpA[s] * a * a / HBARC / HBARC / HBARC / HBARC;
    }
    __shared__ double w[7][IPG_BLOCK / 64];
#pragma unroll
    for (int k = 0; k < 7; k++) {
        double r = wsum(v[k]);
        if ((threadIdx.x & 63) == 0) w[k][threadIdx.x >> 6] = r;
    }
    __syncthreads();
    if (threadIdx.x < 7) {
        double r = 0.;
        for (int q = 0; q < IPG_BLOCK / 64; q++) r += w[threadIdx.x][q];
        ev.partial[(long long)threadIdx.x * ev.nblocks + lb] = r;
    }
}

__global__ __launch_bounds__(IPG_BLOCK) void k_stats_finish(const EvDesc* __restrict__ evs, int nev,
                                                           double* __restrict__ out) {
    const EvDesc& ev = evs[blockIdx.x];
    if (!ev.active) return;
    __shared__ double w[IPG_BLOCK / 64];
    for (int k = 0; k < 7; k++) {
        double acc = 0.;
        for (int b = threadIdx.x; b < ev.nblocks; b += IPG_BLOCK) acc += ev.partial[(long long)k * ev.nblocks + b];
        acc = wsum(acc);
        if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = acc;
        __syncthreads();
        if (threadIdx.x == 0) {
            double r = 0.;
            for (int q = 0; q < IPG_BLOCK / 64; q++) r += w[q];
            out[8 * blockIdx.x + k] = r;
        }
        __syncthreads();
    }
}

// ---- setV: LDS-staged 2D FFT ------------------------------------------------------
// A launch covers a chunk of kc slices [k0, k0+kc) of every event of one
// lattice size N (a template argument: the transform plan is compile-time).
// fftbuf holds [nucleus][slice in chunk][4 packed pairs][S] complex values,
// rows in natural order.

// rows forward: generate rho for row i of (nucleus n, slice k), 4 packed
// complex rows, forward transform along y
// WAVE: 4 wavefronts (BLK = 256), each transforms one of the four packed
// rows, synchronising itself only
// TWL: the twiddle table copied into LDS first (LDS reads in the stages
// instead of global ones)
// RPB: lattice rows a block takes (1 with WAVE); below N = 256 several, so that
// every thread of the block has a site and a butterfly (at N = 128 one row
// gave 128 of 256 threads a site and 64 a radix-8 butterfly: 18.7 -> 15.9 us a
// chunk)
constexpr int setv_rows_per_block(int N) {
    int r = 1;
    while (2 * r * N <= 256 && N % (2 * r) == 0) r *= 2;
    return r;
}
template <int N, int BLK = IPG_BLOCK, bool WAVE = false, bool TWL = false, int RPB = 1>
__global__ __launch_bounds__(BLK) void k_setv_rows_fwd(const EvDesc* __restrict__ evs, FftPlanDev pl, int k0,
                                                      int kc) {
    static_assert(N % RPB == 0 && (!WAVE || RPB == 1), "rows per block");
    __shared__ double2 lds[ipgfft::lds_slots(N, 4 * RPB)];
    __shared__ double2 tws[TWL ? N : 1];
    constexpr int NR = N / RPB;
    const int per_ev = 2 * kc * NR;
    const int e = blockIdx.x / per_ev;
    const int rem = blockIdx.x - e * per_ev;
    const int n = rem / (kc * NR);
    const int kk = (rem / NR) % kc;
    const int i = (rem % NR) * RPB;
    const int k = k0 + kk;
    const EvDesc& ev = evs[e];
    if (!ev.active || k >= ev.Ny) return;
    const size_t S = ev.S;
    const double* g2 = n ? ev.g2B : ev.g2A;
    for (int q = threadIdx.x; q < RPB * N; q += BLK) {
        const int r = RPB == 1 ? 0 : q / N, j = q - r * N;
        const size_t s = (size_t)i * N + q;
        double z[8];
        if (ev.znorm) {
            const double* zp = ev.znorm + (((size_t)n * ev.Ny + k) * S + s) * 8;
#pragma unroll
            for (int c = 0; c < 8; c++) z[c] = zp[c];
        } else {
            normals8(ev.rho_seed, (uint32_t)k, (uint32_t)n, (uint32_t)s, z);
        }
        const double amp = ev.g * sqrt(g2[s] / (double)ev.Ny);
#pragma unroll
        for (int p = 0; p < 4; p++)
            lds[ipgfft::at(N, 4 * r + p, j)] = make_double2(amp * z[2 * p], amp * z[2 * p + 1]);
    }
    const double2* tw = pl.tw;
    if constexpr (TWL) {
        for (int m = threadIdx.x; m < N; m += BLK) tws[m] = pl.tw[m];
        tw = tws;
    }
    __syncthreads();
    if constexpr (WAVE) {
        static_assert(BLK == 256, "one wavefront per packed row");
        ipgfft::wave_fft<N, 1, false>(lds + ipgfft::at(N, (int)(threadIdx.x >> 6), 0), tw);
        __syncthreads();
    } else {
        ipgfft::lds_fft<N, 4 * RPB, BLK, false>(lds, tw);
    }
    double2* out = ev.fftbuf + ((size_t)n * kc + kk) * 4 * S + (size_t)i * N;
    for (int q = threadIdx.x; q < 4 * RPB * N; q += BLK) {
        const int p = q / (RPB * N), t = q - p * (RPB * N), r = RPB == 1 ? 0 : t / N;
        out[(size_t)p * S + t] = lds[ipgfft::at(N, 4 * r + p, t - r * N)];
    }
}

// columns: forward transform, multiply by 1/(k^2+m^2) e^{-|k| UVdamp} / N^2,
// inverse transform; C columns per block.  WAVE: BLK = 64 x (waves), each
// wavefront transforms and filters its own C / waves columns between the
// block's load and store, synchronising itself only.
template <int N, int BLK = IPG_BLOCK, bool WAVE = false>
__global__ __launch_bounds__(BLK) void k_setv_cols(const EvDesc* __restrict__ evs, FftPlanDev pl, int k0, int kc) {
    constexpr int C = ipgfft::cols_per_block(N);
    __shared__ double2 lds[ipgfft::lds_slots(N, C)];
    constexpr int per_pack = N / C;
    const int per_ev = 2 * kc * 4 * per_pack;
    const int e = blockIdx.x / per_ev;
    const int rem = blockIdx.x - e * per_ev;
    const int nk = rem / (4 * per_pack);  // n * kc + kk
    const int p = (rem / per_pack) & 3;
    const int j0 = (rem % per_pack) * C;
    const int k = k0 + nk % kc;
    const EvDesc& ev = evs[e];
    if (!ev.active || k >= ev.Ny) return;
    const size_t S = ev.S;
    double2* buf = ev.fftbuf + ((size_t)nk * 4 + p) * S;
    // load C columns: column c of the block is LDS row c
    for (int q = threadIdx.x; q < C * N; q += blockDim.x) {
        const int r = q / C, c = q - r * C;
        lds[ipgfft::at(N, c, r)] = buf[(size_t)r * N + j0 + c];
    }
    __syncthreads();
    const double m2 = ev.m_lat * ev.m_lat, uv = ev.uvdamp_lat;
    const double invN2 = 1.0 / ((double)N * (double)N);
    auto filter = [&](int c, int r) {
        const double kt2 = pl.s2[r] + pl.s2[j0 + c];
        double f;
        if (m2 == 0.)
            f = kt2 != 0 ? 1. / kt2 : 0.;
        else
            f = (1. / (kt2 + m2)) * exp(-sqrt(kt2) * uv);
        f *= invN2;
        const int a = ipgfft::at(N, c, r);
        lds[a] = make_double2(lds[a].x * f, lds[a].y * f);
    };
    if constexpr (WAVE) {
        constexpr int NW = BLK / 64;
        constexpr int CPW = C / NW;
        static_assert(CPW * NW == C, "columns per wavefront");
        const int w = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
        double2* mine = lds + ipgfft::at(N, w * CPW, 0);
        ipgfft::wave_fft<N, CPW, false>(mine, pl.tw);
        for (int q = lane; q < CPW * N; q += 64) filter(w * CPW + q / N, q % N);
        __syncwarp();
        ipgfft::wave_fft<N, CPW, true>(mine, pl.tw);
        __syncthreads();
    } else {
        ipgfft::lds_fft<N, C, BLK, false>(lds, pl.tw);
        for (int q = threadIdx.x; q < C * N; q += blockDim.x) filter(q / N, q % N);
        __syncthreads();
        ipgfft::lds_fft<N, C, BLK, true>(lds, pl.tw);
    }
    for (int q = threadIdx.x; q < C * N; q += blockDim.x) {
        const int r = q / C, c = q - r * C;
        buf[(size_t)r * N + j0 + c] = lds[ipgfft::at(N, c, r)];
    }
}

// rows inverse for every slice of the chunk in order; each thread keeps the
// Wilson lines of its SPT sites in registers, V <- exp(-i A_k^a t^a) V
// (expq_apply)
template <int N, int kInvBlock, bool TWL = false, int WPE = 1>
__global__ __launch_bounds__(kInvBlock, WPE) void k_setv_rows_inv(const EvDesc* __restrict__ evs, FftPlanDev pl, int k0,
                                                            int kc) {
    constexpr int SPT = (N + kInvBlock - 1) / kInvBlock;
    __shared__ double2 lds[ipgfft::lds_slots(N, 4)];
    __shared__ double2 tws[TWL ? N : 1];
    const int e = blockIdx.x / (2 * N);
    const int n = (blockIdx.x / N) & 1;
    const int i = blockIdx.x % N;
    const EvDesc& ev = evs[e];
    if (!ev.active || k0 >= ev.Ny) return;
    const size_t S = ev.S;
    double* Vg = n ? ev.VB : ev.VA;
    const double2* tw = pl.tw;
    if constexpr (TWL) {
        for (int m = threadIdx.x; m < N; m += kInvBlock) tws[m] = pl.tw[m];
        tw = tws;  // visible after the first barrier of the slice loop
    }
    M3 V[SPT];
#pragma unroll
    for (int t = 0; t < SPT; t++) {
        const int j = threadIdx.x + t * kInvBlock;
        V[t] = j < N ? ldm(Vg, S, (size_t)i * N + j) : m_one();
    }
    const int kend = min(kc, ev.Ny - k0);
    for (int kk = 0; kk < kend; kk++) {
        const double2* in = ev.fftbuf + ((size_t)n * kc + kk) * 4 * S;
        for (int q = threadIdx.x; q < 4 * N; q += blockDim.x) {
            const int p = q / N, j = q - p * N;
            lds[ipgfft::at(N, p, j)] = in[(size_t)p * S + (size_t)i * N + j];
        }
        __syncthreads();
        ipgfft::lds_fft<N, 4, kInvBlock, true>(lds, tw);
#pragma unroll
        for (int t = 0; t < SPT; t++) {
            const int j = threadIdx.x + t * kInvBlock;
            if (j < N) {
                double Q[8];
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    double2 v = lds[ipgfft::at(N, p, j)];
                    Q[2 * p] = -v.x;
                    Q[2 * p + 1] = -v.y;
                }
                ipgad::expq_apply(Q, V[t]);
            }
        }
        __syncthreads();  // the next slice overwrites the LDS rows
    }
#pragma unroll
    for (int t = 0; t < SPT; t++) {
        const int j = threadIdx.x + t * kInvBlock;
        if (j < N) stm(Vg, S, (size_t)i * N + j, V[t]);
    }
}

// this thread's share of the four rows at `in` (plane stride S), value l
// of it at q = threadIdx.x + l BLK (row q / N, element q % N); unrolled by
// recursion, so that every index into `pre` is a constant from the start
// and the array never lands in scratch or LDS
template <int N, int BLK, int L, int l = 0>
__device__ __forceinline__ void setv_fetch_rows(double2 (&pre)[L], const double2* in, size_t S) {
    if constexpr (l < L) {
        const int q = (int)threadIdx.x + l * BLK;
        if (q < 4 * N) {
            const int p = q / N, j = q - p * N;
            pre[l] = in[(size_t)p * S + j];
        }
        setv_fetch_rows<N, BLK, L, l + 1>(pre, in, S);
    }
}
// the same values into the LDS rows
template <int N, int BLK, int L, int l = 0>
__device__ __forceinline__ void setv_put_rows(const double2 (&pre)[L], double2* lds) {
    if constexpr (l < L) {
        const int q = (int)threadIdx.x + l * BLK;
        if (q < 4 * N) {
            const int p = q / N, j = q - p * N;
            lds[ipgfft::at(N, p, j)] = pre[l];
        }
        setv_put_rows<N, BLK, L, l + 1>(pre, lds);
    }
}

// The same pass, software-pipelined: while slice kk is transformed and
// exponentiated, each thread's share of slice kk+1's four rows is already
// on its way into registers, and the twiddles sit in LDS, so that no
// global load inside the loop queues behind that prefetch (vector-memory
// loads retire in order).  WAVE: BLK = 256, each wavefront transforms one
// of the four rows, synchronising itself only.  Same arithmetic as
// k_setv_rows_inv, bit for bit.
template <int N, int BLK, bool WAVE>
__global__ __launch_bounds__(BLK) void k_setv_rows_inv_pf(const EvDesc* __restrict__ evs, FftPlanDev pl, int k0,
                                                         int kc) {
    constexpr int SPT = (N + BLK - 1) / BLK;
    constexpr int L = (4 * N + BLK - 1) / BLK;  // prefetched values per thread
    __shared__ double2 lds[ipgfft::lds_slots(N, 4)];
    __shared__ double2 tws[N];
    const int e = blockIdx.x / (2 * N);
    const int n = (blockIdx.x / N) & 1;
    const int i = blockIdx.x % N;
    const EvDesc& ev = evs[e];
    if (!ev.active || k0 >= ev.Ny) return;
    const size_t S = ev.S;
    for (int m = threadIdx.x; m < N; m += BLK) tws[m] = pl.tw[m];
    double* Vg = n ? ev.VB : ev.VA;
    const int kend = min(kc, ev.Ny - k0);
    const double2* rows = ev.fftbuf + (size_t)n * kc * 4 * S + (size_t)i * N;
    double2 pre[L];
    setv_fetch_rows<N, BLK>(pre, rows, S);
    M3 V[SPT];
#pragma unroll
    for (int t = 0; t < SPT; t++) {
        const int j = threadIdx.x + t * BLK;
        V[t] = j < N ? ldm(Vg, S, (size_t)i * N + j) : m_one();
    }
    for (int kk = 0; kk < kend; kk++) {
        setv_put_rows<N, BLK>(pre, lds);
        if (kk + 1 < kend) setv_fetch_rows<N, BLK>(pre, rows + (size_t)(kk + 1) * 4 * S, S);
        __syncthreads();
        if constexpr (WAVE) {
            static_assert(BLK == 256, "one wavefront per row");
            ipgfft::wave_fft<N, 1, true>(lds + ipgfft::at(N, (int)(threadIdx.x >> 6), 0), tws);
            __syncthreads();
        } else {
            ipgfft::lds_fft<N, 4, BLK, true>(lds, tws);
        }
#pragma unroll
        for (int t = 0; t < SPT; t++) {
            const int j = threadIdx.x + t * BLK;
            if (j < N) {
                double Q[8];
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    double2 v = lds[ipgfft::at(N, p, j)];
                    Q[2 * p] = -v.x;
                    Q[2 * p + 1] = -v.y;
                }
                ipgad::expq_apply(Q, V[t]);
            }
        }
        __syncthreads();  // the next slice overwrites the LDS rows
    }
#pragma unroll
    for (int t = 0; t < SPT; t++) {
        const int j = threadIdx.x + t * BLK;
        if (j < N) stm(Vg, S, (size_t)i * N + j, V[t]);
    }
}

// ---- reverse mode of setV (one event) ---------------------------------------------
// V = E_{Ny-1} ... E_0, E_k = exp(-i A_k^a t^a).  Walking the slices of a chunk
// backwards with the current V and its cotangent Vb in registers:
//   V_k = E_k^+ V,  Eb_k = Vb V_k^+,  Vb <- E_k^+ Vb,  Ab_k = -Qb(Q = -A_k, Eb_k).
// E_k is rebuilt from the Cayley-Hamilton coefficients its reverse needs
// anyway (expq_fcoef: the forward's series below kExpqSeriesMax, its own
// closed form above), equal to the forward's expq_apply to round-off, so
// V_k is recovered to round-off.
// The chunk's A_k are recomputed by the forward row and column passes; Ab_k
// replaces A_k in the transform buffer, row by row.
template <int N, int BLK>
__global__ __launch_bounds__(BLK) void k_adj_setv_rows(const EvDesc* __restrict__ evs, FftPlanDev pl, int k0, int kc,
                                                      double* __restrict__ vv, double* __restrict__ vbar) {
    constexpr int SPT = (N + BLK - 1) / BLK;
    __shared__ double2 lds[ipgfft::lds_slots(N, 4)];
    const int n = blockIdx.x / N;
    const int i = blockIdx.x % N;
    const EvDesc& ev = evs[0];
    if (!ev.active || k0 >= ev.Ny) return;
    const size_t S = ev.S;
    double* Vg = vv + (size_t)n * 18 * S;
    double* Bg = vbar + (size_t)n * 18 * S;
    M3 V[SPT], Vb[SPT];
#pragma unroll
    for (int t = 0; t < SPT; t++) {
        const int j = threadIdx.x + t * BLK;
        V[t] = j < N ? ldm<true>(Vg, S, (size_t)i * N + j) : m_one();
        Vb[t] = j < N ? ldm<true>(Bg, S, (size_t)i * N + j) : m_zero();
    }
    const int kend = min(kc, ev.Ny - k0);
    for (int kk = kend - 1; kk >= 0; kk--) {
        double2* io = ev.fftbuf + ((size_t)n * kc + kk) * 4 * S;
        for (int q = threadIdx.x; q < 4 * N; q += blockDim.x) {
            const int p = q / N, j = q - p * N;
            lds[ipgfft::at(N, p, j)] = io[(size_t)p * S + (size_t)i * N + j];
        }
        __syncthreads();
        ipgfft::lds_fft<N, 4, BLK, true>(lds, pl.tw);
#pragma unroll
        for (int t = 0; t < SPT; t++) {
            const int j = threadIdx.x + t * BLK;
            if (j < N) {
                double Q[8];
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const double2 v = lds[ipgfft::at(N, p, j)];
                    Q[2 * p] = -v.x;
                    Q[2 * p + 1] = -v.y;
                }
                // one set of Cayley-Hamilton coefficients for E and its reverse
                ipgad::ExpQ x;
                ipgad::expq_prep(Q, x);
                const M3 E = ipgad::expq_value(x);
                const M3 Vk = mul_ad(E, V[t]);
                const M3 Eb = mul_bd(Vb[t], Vk);
                Vb[t] = mul_ad(E, Vb[t]);
                V[t] = Vk;
                double Qb[8];
                ipgad::expq_back(x, Eb, Qb);
#pragma unroll
                for (int p = 0; p < 4; p++)
                    io[(size_t)p * S + (size_t)i * N + j] = make_double2(-Qb[2 * p], -Qb[2 * p + 1]);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int t = 0; t < SPT; t++) {
        const int j = threadIdx.x + t * BLK;
        if (j < N) {
            stm<true>(Vg, S, (size_t)i * N + j, V[t]);
            stm<true>(Bg, S, (size_t)i * N + j, Vb[t]);
        }
    }
}

// the Poisson filter is a real, even convolution (self-adjoint): Ab -> rhob
// by the same row / column / row passes; rows forward from the buffer
template <int N>
__global__ __launch_bounds__(IPG_BLOCK) void k_adj_filter_rows_fwd(const EvDesc* __restrict__ evs, FftPlanDev pl,
                                                                  int k0, int kc) {
    __shared__ double2 lds[ipgfft::lds_slots(N, 4)];
    const int per_n = kc * N;
    const int n = blockIdx.x / per_n;
    const int kk = (blockIdx.x / N) % kc;
    const int i = blockIdx.x % N;
    const EvDesc& ev = evs[0];
    if (!ev.active || k0 + kk >= ev.Ny) return;
    const size_t S = ev.S;
    double2* io = ev.fftbuf + ((size_t)n * kc + kk) * 4 * S;
    for (int q = threadIdx.x; q < 4 * N; q += blockDim.x) {
        const int p = q / N, j = q - p * N;
        lds[ipgfft::at(N, p, j)] = io[(size_t)p * S + (size_t)i * N + j];
    }
    __syncthreads();
    ipgfft::lds_fft<N, 4, IPG_BLOCK, false>(lds, pl.tw);
    for (int q = threadIdx.x; q < 4 * N; q += blockDim.x) {
        const int p = q / N, j = q - p * N;
        io[(size_t)p * S + (size_t)i * N + j] = lds[ipgfft::at(N, p, j)];
    }
}
// rows inverse: rhob for colours (2p, 2p+1) = (Re, Im) of packed field p into
// grad[n][k][s][8]
template <int N>
__global__ __launch_bounds__(IPG_BLOCK) void k_adj_filter_rows_inv(const EvDesc* __restrict__ evs, FftPlanDev pl,
                                                                  int k0, int kc, double* __restrict__ grad) {
    __shared__ double2 lds[ipgfft::lds_slots(N, 4)];
    const int per_n = kc * N;
    const int n = blockIdx.x / per_n;
    const int kk = (blockIdx.x / N) % kc;
    const int i = blockIdx.x % N;
    const EvDesc& ev = evs[0];
    const int k = k0 + kk;
    if (!ev.active || k >= ev.Ny) return;
    const size_t S = ev.S;
    const double2* in = ev.fftbuf + ((size_t)n * kc + kk) * 4 * S;
    for (int q = threadIdx.x; q < 4 * N; q += blockDim.x) {
        const int p = q / N, j = q - p * N;
        lds[ipgfft::at(N, p, j)] = in[(size_t)p * S + (size_t)i * N + j];
    }
    __syncthreads();
    ipgfft::lds_fft<N, 4, IPG_BLOCK, true>(lds, pl.tw);
    for (int j = threadIdx.x; j < N; j += blockDim.x) {
        double* g = grad + (((size_t)n * ev.Ny + k) * S + (size_t)i * N + j) * 8;
#pragma unroll
        for (int p = 0; p < 4; p++) {
            g[2 * p] = lds[ipgfft::at(N, p, j)].x;
            g[2 * p + 1] = lds[ipgfft::at(N, p, j)].y;
        }
    }
}

__global__ __launch_bounds__(IPG_BLOCK) void k_unit_v(const EvDesc* __restrict__ evs, int nev) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active) return;
    const long long s = (long long)xcd_remap(blockIdx.x - ev.block0, ev.nblocks) * IPG_BLOCK + threadIdx.x;
    if (s >= ev.S) return;
    stm(ev.VA, ev.S, s, m_one());
    stm(ev.VB, ev.S, s, m_one());
}

__global__ void k_rho_normals(const EvDesc* __restrict__ evs, int nucleus, int k, double* out) {
    const EvDesc& ev = evs[0];
    long long s = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= ev.S) return;
    double z[8];
    normals8(ev.rho_seed, (uint32_t)k, (uint32_t)nucleus, (uint32_t)s, z);
    for (int c = 0; c < 8; c++) out[8 * s + c] = z[c];
}

// ---- links (Init.cpp:2459-2491) ------------------------------------------------
__device__ __forceinline__ M3 ld_guarded(const double* V, size_t S, size_t s) {
    M3 m = ldm(V, S, s);
    cd t = tr(m);
    if (t.r != t.r || t.i != t.i) m = m_one();
    return m;
}

__global__ __launch_bounds__(IPG_BLOCK) void k_links(const EvDesc* __restrict__ evs, int nev) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active) return;
    const long long s = (long long)xcd_remap(blockIdx.x - ev.block0, ev.nblocks) * IPG_BLOCK + threadIdx.x;
    if (s >= ev.S) return;
    const int N = ev.N;
    const size_t S = ev.S;
    const int i = (int)(s / N), j = (int)(s - (long long)i * N);
    const size_t pX = (size_t)clampi(i + 1, N) * N + j, pY = (size_t)i * N + clampi(j + 1, N);
    M3 va = ld_guarded(ev.VA, S, s), vb = ld_guarded(ev.VB, S, s);
    stm(ev.L1x, S, s, mul_bd(va, ld_guarded(ev.VA, S, pX)));
    stm(ev.L1y, S, s, mul_bd(va, ld_guarded(ev.VA, S, pY)));
    stm(ev.L2x, S, s, mul_bd(vb, ld_guarded(ev.VB, S, pX)));
    stm(ev.L2y, S, s, mul_bd(vb, ld_guarded(ev.VB, S, pY)));
}

// ---- tau = 0 root finder (Init.cpp:3344-3481) ------------------------------------
constexpr int NWB = 64;  // one wavefront per block: the Jacobian lives in LDS

__device__ __forceinline__ void restart_alpha(uint64_t seed, uint32_t link, uint32_t draw, double al[8]) {
    normals8(seed, draw, 0xFFFF0000u, link, al);
}

// F_a = -Im[tr t^a (W - W^+) + tr t^a (W U^+ - U W^+)]; trci[a] is the first
// trace.  The second matrix is W U^+ minus its own conjugate, so one product
// gives both; returns sum |F_a|
__device__ __forceinline__ double residual(const M3& W, const M3& Us, const double (&trci)[8], double (&F)[8]) {
    const AH m = ah_of(mul_bd(W, Us));
    const double s3 = 1.0 / (2.0 * sqrt(3.0));
    const double t[8] = {m.o[0].i, m.o[0].r, 0.5 * (m.d[0] - m.d[1]), m.o[1].i, m.o[1].r, m.o[2].i, m.o[2].r,
                         s3 * (m.d[0] + m.d[1]) - 2.0 * s3 * m.d[2]};
    double Fz = 0.;
#pragma unroll
    for (int a = 0; a < 8; a++) {
        F[a] = -(trci[a] + t[a]);
        Fz += fabs(F[a]);
    }
    return Fz;
}
// the finite-difference steps and the exponent of Jacobian column c: the
// serial loop adds the step to alpha[b] and subtracts it again in place, so
// column c sees (alpha[k] + d_k) - d_k for k < c; returns d_c
__device__ __forceinline__ double column_exponent(const double (&alpha)[8], int c, double (&p)[8]) {
    double d = 0.;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const double dk = fmax(0.001, fmin(10., 0.01 * fabs(alpha[k])));
        p[k] = k < c ? (alpha[k] + dk) - dk : (k == c ? alpha[k] + dk : alpha[k]);
        if (k == c) d = dk;
    }
    return d;
}
// the column 2 Im tr t^a W D / d, D = (E - Us)^+; false where the reference's running
// sum |J_a| stays below 1e-15 (it then takes the analytic Jacobian)
__device__ __forceinline__ bool jacobian_column(const M3& W, const M3& D, double d, double (&col)[8]) {
    const M3 Mp = W * D;
    cd t[8];
    tr_gen(Mp, t);
    double chk = 0.;
    bool good = true;
#pragma unroll
    for (int a = 0; a < 8; a++) {
        col[a] = 2. * t[a].i / d;
        chk += fabs(col[a]);
        if (chk < 1e-15) good = false;
    }
    return good;
}
// the analytic column about U = Us
__device__ __forceinline__ void analytic_column(const M3& W, const M3& Us, int c, double (&col)[8]) {
    const M3 Mb = gen_mul(c, dag(Us));
#pragma unroll
    for (int a = 0; a < 8; a++) col[a] = -2. * retrprod(gen_mul(a, W), Mb);
}
// First pass of the root finder: four lanes per link, 16 links a wavefront.
// Each lane evaluates two Jacobian columns; the system goes through LDS and
// every lane solves it in registers.  The first iteration starts from exponent
// 0 at every link, so its column exponentials are the same everywhere and come
// from a table.  Almost every link converges in two to six iterations (mean
// 2.1 to 4.0 over the lattices in use); one that has not after kQuadIter, or
// that wants a restart, goes to its event's list for k_newton, which starts it
// afresh.
// FP64 issue bounds it, most of it in the exponentials.  N = 512 (2.1
// iterations a link) / N = 128 (3.2): eight lanes a link, all of them repeating
// the residual, the update and its exponential, with the elimination by
// shuffles 1740 / 380 us; this 1020 + 244 / 98 + 9 us (both passes).  Two
// lanes a link with the columns in registers is less work, but spills at two
// waves per SIMD (1324 / 190 us).
constexpr int kQuadIter = 8;
constexpr int kQuadLinks = 16;
__global__ __launch_bounds__(64, 2) void k_newton_quad(const EvDesc* __restrict__ evs, int nev, int* __restrict__ cnt) {
    __shared__ double mU0[18][kQuadLinks], mW[18][kQuadLinks], mUs[18][kQuadLinks];
    __shared__ double mJ[64][kQuadLinks];  // row-major
    __shared__ double tab[8][18];          // exp(i d t^c), d the first step
    const int lane = threadIdx.x;
    const int sub = lane & 3, k = lane >> 2;
    constexpr int kPer = NWB / kQuadLinks;  // blocks per 64-link block
    const int e = find_event_links(evs, nev, (int)blockIdx.x / kPer);
    const EvDesc& ev = evs[e];
    if (!ev.active) return;
    const long long S = ev.S;
    const long long l = ((long long)blockIdx.x - (long long)kPer * ev.lblock0) * kQuadLinks + k;
    // 2 S is a multiple of 512: a block is full or past the end
    if (l - k >= 2 * S) return;
    const int dir = l >= S;
    const long long s = dir ? l - S : l;
    auto ld = [&](const double (*m)[kQuadLinks]) {
        // read where used: kept in registers across the loops they spill
        asm volatile("" ::: "memory");
        M3 r;
#pragma unroll
        for (int q = 0; q < 9; q++) r.e[q] = cd{m[2 * q][k], m[2 * q + 1][k]};
        return r;
    };
    auto st = [&](double (*m)[kQuadLinks], const M3& r) {
#pragma unroll
        for (int q = 0; q < 9; q++) {
            m[2 * q][k] = r.e[q].r;
            m[2 * q + 1][k] = r.e[q].i;
        }
    };
    double alpha[8];
#pragma unroll
    for (int a = 0; a < 8; a++) alpha[a] = 0.;
    if (lane < 8) {
        double p[8];
        (void)column_exponent(alpha, lane, p);
        const M3 E = exp_iQt(p);
#pragma unroll
        for (int q = 0; q < 9; q++) {
            tab[lane][2 * q] = E.e[q].r;
            tab[lane][2 * q + 1] = E.e[q].i;
        }
    }
    const M3 U1 = ldm(dir ? ev.L1y : ev.L1x, S, s);
    const M3 U2 = ldm(dir ? ev.L2y : ev.L2x, S, s);
    if (sub == 0) {
        const M3 U0 = U1 * U2;
        st(mU0, U0);
        st(mW, U1 + U2);
        // exp(0) is the identity (its closed form gives no number, the guard 1)
        st(mUs, U0);
    }
    bool done = false, failed = false;
    int analytic = 0;
    __syncthreads();
    for (int iter = 1; iter <= kQuadIter && __any(!done); iter++) {
        // not unrolled: one copy of the exponential keeps the kernel inside the
        // instruction cache
        bool good = true;
#pragma unroll 1
        for (int q = 0; q < 2; q++) {
            const int c = 2 * sub + q;
            double p[8], col[8];
            const double d = column_exponent(alpha, c, p);
            M3 E;
            if (iter == 1) {
#pragma unroll
                for (int r = 0; r < 9; r++) E.e[r] = cd{tab[c][2 * r], tab[c][2 * r + 1]};
            } else {
                E = exp_iQt(p);
            }
            E = E * ld(mU0);
            E = dag(E) - dag(ld(mUs));
            good = jacobian_column(ld(mW), E, d, col) && good;
#pragma unroll
            for (int a = 0; a < 8; a++) mJ[8 * a + c][k] = col[a];
        }
        const unsigned long long bad = __ballot(!good);
        if ((bad >> (lane & ~3)) & 15ull) {
            analytic = 1;
#pragma unroll 1
            for (int q = 0; q < 2; q++) {
                double col[8];
                analytic_column(ld(mW), ld(mUs), 2 * sub + q, col);
#pragma unroll
                for (int a = 0; a < 8; a++) mJ[8 * a + 2 * sub + q][k] = col[a];
            }
        }
        double F[8];
        double Fzero;
        {
            const M3 W = ld(mW);
            cd trc[8];
            tr_gen(W - dag(W), trc);
            double trci[8];
#pragma unroll
            for (int a = 0; a < 8; a++) trci[a] = trc[a].i;
            Fzero = residual(W, ld(mUs), trci, F);
        }
        __syncthreads();
        {
            double J[64];
#pragma unroll
            for (int a = 0; a < 64; a++) J[a] = mJ[a][k];
            solve_rows(J, F);
        }
        bool okstep = true;
#pragma unroll
        for (int a = 0; a < 8; a++) {
            if (fabs(F[a]) > 1e5) okstep = false;
            const double dk = fmax(0.001, fmin(10., 0.01 * fabs(alpha[a])));
            alpha[a] = ((alpha[a] + dk) - dk) + F[a];
        }
        M3 Us = exp_iQt(alpha);
        Us = Us * ld(mU0);
        __syncthreads();
        if (sub == 0 && !done) st(mUs, Us);
        if (!done) {
            if (!okstep) {
                done = failed = true;
            } else if (!(Fzero > 1e-6)) {
                done = true;
                if (sub == 0) {
                    stm(ev.U[0][dir], S, s, Us);
                    ev.newton_stat[l] = iter | (analytic << 29);
                }
            }
        }
        __syncthreads();
    }
    if (!done) failed = true;
    // unfinished links, one entry each
    const unsigned long long m = __ballot(failed && sub == 0);
    if (m) {
        const int first = __ffsll((long long)m) - 1;
        int base = 0;
        if (lane == first) base = atomicAdd(&cnt[1 + e], __popcll(m));
        base = __shfl(base, first, 64);
        if (failed && sub == 0)
            ((int*)ev.land_epsv)[base + __popcll(m & ((1ull << lane) - 1ull))] = (int)l;
    }
}

// The links k_newton_quad leaves, one per group of NG = 8 lanes
// (Init.cpp:3386-3476): a few links in a million take tens to thousands of
// iterations, so here the latency of an iteration counts.  Lane c of a group
// evaluates Jacobian column c (one SU(3) exponential); every lane carries the
// same link state and computes the residual, the elimination (in registers:
// through shuffles it was a third of the iteration), the update and the next
// iterate redundantly.  A group takes its next link from a wave-aggregated
// work counter as soon as its link is done.
constexpr int NG = 8;

__device__ __forceinline__ M3 lds_m3(const double* p) {
    M3 m;
#pragma unroll
    for (int k = 0; k < 9; k++) m.e[k] = cd{p[2 * k], p[2 * k + 1]};
    return m;
}
__device__ __forceinline__ void lds_st(double* p, const M3& m) {
#pragma unroll
    for (int k = 0; k < 9; k++) {
        p[2 * k] = m.e[k].r;
        p[2 * k + 1] = m.e[k].i;
    }
}

// exp(i best t) U0, or the identity, into out; out of line: 200 restarts without
// a root are rare
__device__ __attribute__((noinline)) void best_iterate(const double* best, const double* U0, int one, double* out) {
    double ba[8];
#pragma unroll
    for (int a = 0; a < 8; a++) ba[a] = best[a];
    lds_st(out, one ? m_one() : exp_iQt(ba) * lds_m3(U0));
}

// cnt[0]: the work counter, cnt[1 + e]: the length of event e's list
__global__ __launch_bounds__(NWB, 1) void k_newton(const EvDesc* __restrict__ evs, int nev, int* __restrict__ cnt) {
    __shared__ double Jt[NWB / NG][8][8];  // [group][row a][column c]
    // per group: U0 = U1 U2, W = U1 + U2, the iterate Us (written by lane 0)
    __shared__ double Ms[NWB / NG][3][18];
    __shared__ double Bs[NWB / NG][16];    // best exponent, Im tr t^a (W - W^+)
    const int lane = threadIdx.x;
    const int c = lane & (NG - 1);
    const int grp = lane / NG;
    const int maxIt = 2000, maxRe = 200;
    double* mU0 = Ms[grp][0];
    double* mW = Ms[grp][1];
    double* mUs = Ms[grp][2];
    double* best_alpha = Bs[grp];
    double* trci = Bs[grp] + 8;
    int state = 0;  // group-uniform: 0 needs a link, 1 iterating, 2 no work left
    int e = 0, dir = 0;
    long long l = 0, s = 0;
    uint32_t link = 0;
    double alpha[8];
#pragma unroll
    for (int a = 0; a < 8; a++) alpha[a] = 0.;
    double Fzero = 0., Fmin = 0.;
    int iter = 0, nRestart = 0, total = 0, analytic = 0, best_one = 1;
    uint32_t ndraw = 0;
    if (c == 0) {
        lds_st(mU0, m_one());
        lds_st(mW, m_one());
        lds_st(mUs, m_one());
#pragma unroll
        for (int a = 0; a < 16; a++) Bs[grp][a] = 0.;
    }
    for (;;) {
        // ---- one request per idle group
        const bool lead_need = state == 0 && c == 0;
        const unsigned long long need = __ballot(lead_need);
        if (need) {
            const int first = __ffsll((long long)need) - 1;
            int base = 0;
            if (lane == first) base = atomicAdd(cnt, __popcll(need));
            base = __shfl(base, first, NWB);
            int g = lead_need ? base + __popcll(need & ((1ull << lane) - 1ull)) : 0;
            g = __shfl(g, 0, NG);
            if (state == 0) {
                // entry g of the events' lists, one after the other
                e = 0;
                while (e < nev && g >= cnt[1 + e]) g -= cnt[1 + e++];
                if (e >= nev) {
                    state = 2;
                    e = 0;
                } else {
                    const EvDesc& ev = evs[e];
                    const long long S = ev.S;
                    l = ((const int*)ev.land_epsv)[g];
                    {
                        dir = l >= S;
                        s = dir ? l - S : l;
                        link = (uint32_t)(2 * s + dir);
#pragma unroll
                        for (int a = 0; a < 8; a++) alpha[a] = 0.;
                        if (c == 0) {
                            const M3 U1 = ldm(dir ? ev.L1y : ev.L1x, S, s);
                            const M3 U2 = ldm(dir ? ev.L2y : ev.L2x, S, s);
                            const M3 U0 = U1 * U2;
                            const M3 W = U1 + U2;
                            cd trc[8];
                            tr_gen(W - dag(W), trc);
#pragma unroll
                            for (int a = 0; a < 8; a++) trci[a] = trc[a].i;
                            lds_st(mU0, U0);
                            lds_st(mW, W);
                            // exp(0) is the identity (its closed form gives no number, the guard 1)
                            lds_st(mUs, U0);
                        }
                        best_one = 1;
                        Fzero = 10.;
                        Fmin = 1e6;
                        iter = nRestart = total = analytic = 0;
                        ndraw = 0;
                        state = 1;
                    }
                }
            }
        }
        if (__ballot(state != 2) == 0) break;
        __syncthreads();  // link state written by lane 0 of each group

        // ---- one iteration; every group runs it (uniform control flow for
        // the barriers), only groups in state 1 keep the result
        iter++;
        total++;
        double F[8];
        {
            double tr8[8];
#pragma unroll
            for (int a = 0; a < 8; a++) tr8[a] = trci[a];
            Fzero = residual(lds_m3(mW), lds_m3(mUs), tr8, F);
        }
        double col[8];
        double p[8];
        const double d = column_exponent(alpha, c, p);
        const bool good = jacobian_column(lds_m3(mW), dag(exp_iQt(p) * lds_m3(mU0)) - dag(lds_m3(mUs)), d, col);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const double dk = fmax(0.001, fmin(10., 0.01 * fabs(alpha[k])));
            alpha[k] = (alpha[k] + dk) - dk;
        }
        const unsigned long long bad = __ballot(!good);
        if ((bad >> (grp * NG)) & 0xFFull) {
            analytic = 1;
            analytic_column(lds_m3(mW), lds_m3(mUs), c, col);
        }
        // ---- the columns of the group's lanes
#pragma unroll
        for (int a = 0; a < 8; a++) Jt[grp][a][c] = col[a];
        __syncthreads();
        double J[64];
#pragma unroll
        for (int k = 0; k < 64; k++) J[k] = Jt[grp][k >> 3][k & 7];
        __syncthreads();
        solve_rows(J, F);
        double(&y)[8] = F;
        bool okstep = true;
#pragma unroll
        for (int a = 0; a < 8; a++)
            if (fabs(y[a]) > 1e5) okstep = false;
        if (okstep) {
#pragma unroll
            for (int a = 0; a < 8; a++) alpha[a] = alpha[a] + y[a];
        } else {
            restart_alpha(evs[e].newton_seed, link, ndraw++, alpha);
        }
        if (Fzero < Fmin) {
            // best = the new iterate, kept as its exponent (Us is exp(i alpha t) U0)
            Fmin = Fzero;
            if (c == 0)
#pragma unroll
                for (int a = 0; a < 8; a++) best_alpha[a] = alpha[a];
            best_one = 0;
        }
        if (iter == maxIt) {
            restart_alpha(evs[e].newton_seed, link, ndraw++, alpha);
            nRestart++;
            iter = 0;
        }
        M3 Us = exp_iQt(alpha) * lds_m3(mU0);
        if (c == 0) lds_st(mUs, Us);
        const bool stop = state == 1 && !(Fzero > 1e-6 && iter < maxIt && nRestart < maxRe);
        if (stop) {
            const EvDesc& ev = evs[e];
            const int conv = nRestart != maxRe;
            if (c == 0) {
                if (!conv) {
                    best_iterate(best_alpha, mU0, best_one, mUs);
                    Us = lds_m3(mUs);
                }
                stm(ev.U[0][dir], ev.S, s, Us);
                ev.newton_stat[l] = total | (nRestart << 20) | ((!conv) << 28) | (analytic << 29);
            }
            state = 0;
        }
        __syncthreads();  // Us, best exponent visible before the next round
    }
}

// newton_polish: exact Newton steps of the converged links, U <- exp(i y^a t^a) U
// with J_ab = -2 Re tr(t^a W U^+ t^b) about U.  A lane a link, everything in
// registers: no work is repeated and every link takes the same steps (in
// k_newton, where the polishing links were, eight lanes repeat the elimination
// and the exponential of a link and no more than 1024 wavefronts run: the tau = 0
// fields with four steps took 7.8 ms at N = 512 and 2.5 at N = 256; with this
// kernel 1.31 and 0.50, without steps 1.15 and 0.46).
__global__ __launch_bounds__(NWB, 1) void k_newton_polish(const EvDesc* __restrict__ evs, int nev) {
    const int e = find_event_links(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active || ev.newton_polish == 0) return;
    const long long S = ev.S;
    const long long l = ((long long)blockIdx.x - ev.lblock0) * NWB + threadIdx.x;
    if (l >= 2 * S) return;
    const int dir = l >= S;
    const long long s = dir ? l - S : l;
    const int stat = ev.newton_stat[l];
    if (stat & (1 << 28)) return;  // no root found
    const M3 W = ldm(dir ? ev.L1y : ev.L1x, S, s) + ldm(dir ? ev.L2y : ev.L2x, S, s);
    M3 Us = ldm(ev.U[0][dir], S, s);
    double trci[8];
    {
        cd trc[8];
        tr_gen(W - dag(W), trc);
#pragma unroll
        for (int a = 0; a < 8; a++) trci[a] = trc[a].i;
    }
    // a step that finds the residual above the stopping level is not counted
    int total = 0;
    for (int n = 0; n < ev.newton_polish && total < 2000; total++) {
        double F[8];
        if (!(residual(W, Us, trci, F) > 1e-6)) n++;
        const M3 UW = mul_bd(Us, W);
        double J[64];
#pragma unroll
        for (int c = 0; c < 8; c++) {
            cd t[8];
            tr_gen(dag(gen_mul(c, UW)), t);
#pragma unroll
            for (int a = 0; a < 8; a++) J[8 * a + c] = -2. * t[a].r;
        }
        solve_rows(J, F);
        Us = exp_step(F) * Us;
    }
    stm(ev.U[0][dir], S, s, Us);
    ev.newton_stat[l] = stat + total;
}

// A^eta from the four links touching the site, pi = -(2i/g) A^eta
__global__ __launch_bounds__(IPG_BLOCK) void k_pi_init(const EvDesc* __restrict__ evs, int nev) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active) return;
    const long long s = (long long)xcd_remap(blockIdx.x - ev.block0, ev.nblocks) * IPG_BLOCK + threadIdx.x;
    if (s >= ev.S) return;
    const int N = ev.N;
    const size_t S = ev.S;
    const int i = (int)(s / N), j = (int)(s - (long long)i * N);
    const size_t mX = (size_t)clampi(i - 1, N) * N + j, mY = (size_t)i * N + clampi(j - 1, N);
    M3 acc;
    {
        M3 D = ldm(ev.L1x, S, s) - ldm(ev.L2x, S, s);
        M3 Dd = dag(D);
        M3 U = ldm(ev.U[0][0], S, s);
        acc = ((mul_bd(D, U) - D) - U * Dd) + Dd;
        D = ldm(ev.L1x, S, mX) - ldm(ev.L2x, S, mX);
        Dd = dag(D);
        U = ldm(ev.U[0][0], S, mX);
        acc = (((acc - mul_ad(U, D)) + D) + Dd * U) - Dd;
    }
    {
        M3 D = ldm(ev.L1y, S, s) - ldm(ev.L2y, S, s);
        M3 Dd = dag(D);
        M3 U = ldm(ev.U[0][1], S, s);
        acc = (((acc + mul_bd(D, U)) - D) - U * Dd) + Dd;
        D = ldm(ev.L1y, S, mY) - ldm(ev.L2y, S, mY);
        Dd = dag(D);
        U = ldm(ev.U[0][1], S, mY);
        acc = (((acc - mul_ad(U, D)) + D) + Dd * U) - Dd;
    }
    // pi = (-2i/g) (1/8) acc
    sth(ev.pi, S, s, mul_i(-2. / ev.g, (1. / 8.) * acc));
}

__global__ __launch_bounds__(IPG_BLOCK) void k_zero_fields(const EvDesc* __restrict__ evs, int nev) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active) return;
    const long long s = (long long)xcd_remap(blockIdx.x - ev.block0, ev.nblocks) * IPG_BLOCK + threadIdx.x;
    if (s >= ev.S) return;
    const M3 z = m_zero();
    sth(ev.E1, ev.S, s, z);
    sth(ev.E2, ev.S, s, z);
    sth(ev.phi[0], ev.S, s, z);
}

}  // namespace

void ipg_launch_tp(const EvDesc* d, int nev, int nblk, hipStream_t st) {
    hipLaunchKernelGGL(k_tp_g, dim3(nblk), dim3(IPG_BLOCK), 0, st, d, nev);
    hipLaunchKernelGGL(k_tp, dim3(nblk), dim3(IPG_BLOCK), 0, st, d, nev);
}
void ipg_launch_qs(const EvDesc* d, int nev, int nblk, const double* Tl, const double* Q, int* flag,
                   hipStream_t st) {
    hipLaunchKernelGGL(k_qs_b, dim3(nblk), dim3(IPG_BLOCK), 0, st, d, nev, Tl, Q, flag);
    hipLaunchKernelGGL(k_qs_a, dim3(nblk), dim3(IPG_BLOCK), 0, st, d, nev, Tl, Q, flag);
    hipLaunchKernelGGL(k_qs_serial, dim3(nev), dim3(64), 0, st, d, nev, Tl, Q, (const int*)flag);
}
void ipg_launch_stats(const EvDesc* d, int nev, int nblk, double* out, hipStream_t st) {
    hipLaunchKernelGGL(k_stats, dim3(nblk), dim3(IPG_BLOCK), 0, st, d, nev);
    hipLaunchKernelGGL(k_stats_finish, dim3(nev), dim3(IPG_BLOCK), 0, st, d, nev, out);
}
// variants (the same arithmetic in other launch shapes; the autotuner picks
// each): v.inv, v.fwd, v.cols = 0 for 256-thread blocks, 1 for 512-thread
// blocks of the inverse row, forward row and column passes, 2 for the
// wavefront-synchronised transforms of the forward row and column passes;
// v.inv = 2, 3: the prefetching inverse row pass in 512-thread blocks and
// in 256-thread blocks with wavefront-synchronised transforms; v.inv = 4, 5
// and v.fwd = 3: variants 0, 1 and 2 with the twiddles read from LDS (5 held
// to 128 registers, four waves per SIMD).  Below N = 256 the forward row pass
// takes several lattice rows a block (the inverse one, serial in the slices,
// keeps one: two rows a block left half of the CUs without a block, 28 -> 37
// us a chunk at N = 128).  Each pass is bracketed by its pair of events when
// they are given.

// the column pass in the launch shape of variant cv
template <int N>
static void launch_cols(const EvDesc* d, const FftPlanDev& pl, int k0, int kc, int ncol, int cv, hipStream_t st) {
    constexpr int C = ipgfft::cols_per_block(N);
    constexpr int CW = C < 8 ? C : 8;
    if (cv == 1)
        hipLaunchKernelGGL((k_setv_cols<N, 512>), dim3(ncol), dim3(512), 0, st, d, pl, k0, kc);
    else if (cv == 2)
        hipLaunchKernelGGL((k_setv_cols<N, 64 * CW, true>), dim3(ncol), dim3(64 * CW), 0, st, d, pl, k0, kc);
    else
        hipLaunchKernelGGL((k_setv_cols<N, IPG_BLOCK>), dim3(ncol), dim3(IPG_BLOCK), 0, st, d, pl, k0, kc);
}
template <int N>
static void launch_rows_fwd(const EvDesc* d, int nev, const FftPlanDev& pl, int k0, int kc, int v, hipStream_t st) {
    constexpr int R = setv_rows_per_block(N);
    const dim3 g((unsigned)(nev * 2 * kc * (N / R)));
    if constexpr (N >= 256) {
        if (v == 1) {
            hipLaunchKernelGGL((k_setv_rows_fwd<N, 512>), g, dim3(512), 0, st, d, pl, k0, kc);
            return;
        }
        if (v == 2) {
            hipLaunchKernelGGL((k_setv_rows_fwd<N, 256, true>), g, dim3(256), 0, st, d, pl, k0, kc);
            return;
        }
        if (v == 3) {
            hipLaunchKernelGGL((k_setv_rows_fwd<N, 256, true, true>), g, dim3(256), 0, st, d, pl, k0, kc);
            return;
        }
    }
    hipLaunchKernelGGL((k_setv_rows_fwd<N, IPG_BLOCK, false, false, R>), g, dim3(IPG_BLOCK), 0, st, d, pl, k0, kc);
}
template <int N>
static void setv_chunk(const EvDesc* d, int nev, const FftPlanDev& pl, int k0, int kc, const SetvVariant& v,
                       const SetvEvents& t, hipStream_t st) {
    constexpr int C = ipgfft::cols_per_block(N);
    const int ncol = nev * 2 * kc * 4 * (N / C);
    const int nrow_inv = nev * 2 * N;
    const int inv_variant = v.inv;
    const hipEvent_t ev_a = t.inv[0], ev_b = t.inv[1];
    if (t.fwd[0]) (void)hipEventRecord(t.fwd[0], st);
    launch_rows_fwd<N>(d, nev, pl, k0, kc, v.fwd, st);
    if (t.fwd[1]) (void)hipEventRecord(t.fwd[1], st);
    if (t.cols[0]) (void)hipEventRecord(t.cols[0], st);
    launch_cols<N>(d, pl, k0, kc, ncol, v.cols, st);
    if (t.cols[1]) (void)hipEventRecord(t.cols[1], st);
    if (ev_a) (void)hipEventRecord(ev_a, st);
    if (inv_variant == 1)
        hipLaunchKernelGGL((k_setv_rows_inv<N, 512>), dim3(nrow_inv), dim3(512), 0, st, d, pl, k0, kc);
    else if (inv_variant == 2)
        hipLaunchKernelGGL((k_setv_rows_inv_pf<N, 512, false>), dim3(nrow_inv), dim3(512), 0, st, d, pl, k0, kc);
    else if (inv_variant == 3)
        hipLaunchKernelGGL((k_setv_rows_inv_pf<N, 256, true>), dim3(nrow_inv), dim3(256), 0, st, d, pl, k0, kc);
    else if (inv_variant == 4)
        hipLaunchKernelGGL((k_setv_rows_inv<N, 256, true>), dim3(nrow_inv), dim3(256), 0, st, d, pl, k0, kc);
    else if (inv_variant == 5)
        hipLaunchKernelGGL((k_setv_rows_inv<N, 512, true, 4>), dim3(nrow_inv), dim3(512), 0, st, d, pl, k0, kc);
    else
        hipLaunchKernelGGL((k_setv_rows_inv<N, 256>), dim3(nrow_inv), dim3(256), 0, st, d, pl, k0, kc);
    if (ev_b) (void)hipEventRecord(ev_b, st);
}
void ipg_launch_setv_chunk(const EvDesc* d, int nev, const FftPlanDev& pl, int k0, int kc, const SetvVariant& v,
                           const SetvEvents& t, hipStream_t st) {
#define IPG_SETV_CASE(n) \
    case n: setv_chunk<n>(d, nev, pl, k0, kc, v, t, st); break;
    switch (pl.N) {
        IPG_SETV_CASE(16)
        IPG_SETV_CASE(32)
        IPG_SETV_CASE(48)
        IPG_SETV_CASE(64)
        IPG_SETV_CASE(96)
        IPG_SETV_CASE(128)
        IPG_SETV_CASE(192)
        IPG_SETV_CASE(256)
        IPG_SETV_CASE(384)
        IPG_SETV_CASE(512)
        IPG_SETV_CASE(768)
        IPG_SETV_CASE(1024)
        default: break;  // rejected by the engine set-up
    }
#undef IPG_SETV_CASE
}
template <int N>
static void adj_setv_chunk(const EvDesc* d, const FftPlanDev& pl, int k0, int kc, double* vv, double* vbar,
                           double* grad, const SetvVariant& v, hipStream_t st, bool recompute) {
    constexpr int C = ipgfft::cols_per_block(N);
    const int nrow = 2 * kc * N;
    const int ncol = 2 * kc * 4 * (N / C);
    // recompute the chunk's A_k (forward row and column passes) unless the
    // buffer already holds them
    if (recompute) {
        launch_rows_fwd<N>(d, 1, pl, k0, kc, v.fwd, st);
        launch_cols<N>(d, pl, k0, kc, ncol, v.cols, st);
    }
    hipLaunchKernelGGL((k_adj_setv_rows<N, 256>), dim3(2 * N), dim3(256), 0, st, d, pl, k0, kc, vv, vbar);
    hipLaunchKernelGGL(k_adj_filter_rows_fwd<N>, dim3(nrow), dim3(IPG_BLOCK), 0, st, d, pl, k0, kc);
    launch_cols<N>(d, pl, k0, kc, ncol, v.cols, st);
    hipLaunchKernelGGL(k_adj_filter_rows_inv<N>, dim3(nrow), dim3(IPG_BLOCK), 0, st, d, pl, k0, kc, grad);
}
void ipg_adj_setv_chunk(const EvDesc* d, const FftPlanDev& pl, int k0, int kc, double* vv, double* vbar,
                        double* grad, const SetvVariant& v, hipStream_t st, bool recompute) {
#define IPG_ADJ_CASE(n) \
    case n: adj_setv_chunk<n>(d, pl, k0, kc, vv, vbar, grad, v, st, recompute); break;
    switch (pl.N) {
        IPG_ADJ_CASE(16)
        IPG_ADJ_CASE(32)
        IPG_ADJ_CASE(48)
        IPG_ADJ_CASE(64)
        IPG_ADJ_CASE(96)
        IPG_ADJ_CASE(128)
        IPG_ADJ_CASE(192)
        IPG_ADJ_CASE(256)
        IPG_ADJ_CASE(384)
        IPG_ADJ_CASE(512)
        IPG_ADJ_CASE(768)
        IPG_ADJ_CASE(1024)
        default: break;
    }
#undef IPG_ADJ_CASE
}
void ipg_launch_unit_v(const EvDesc* d, int nev, int nblk, hipStream_t st) {
    hipLaunchKernelGGL(k_unit_v, dim3(nblk), dim3(IPG_BLOCK), 0, st, d, nev);
}
void ipg_launch_links(const EvDesc* d, int nev, int nblk, hipStream_t st) {
    hipLaunchKernelGGL(k_links, dim3(nblk), dim3(IPG_BLOCK), 0, st, d, nev);
}
__global__ void k_zero_counters(int* c, int n) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) c[t] = 0;
}

// d_cnt: 1 + nev ints.  The second pass is persistent: enough one-wave blocks
// for a wave on every SIMD (256 CUs x 4); each loops until the lists run out.
void ipg_launch_newton(const EvDesc* d, int nev, int nlinkblk, int* d_cnt, bool polish, hipStream_t st) {
    hipLaunchKernelGGL(k_zero_counters, dim3((unsigned)(nev + 1 + 255) / 256), dim3(256), 0, st, d_cnt, nev + 1);
    hipLaunchKernelGGL(k_newton_quad, dim3(NWB / kQuadLinks * nlinkblk), dim3(NWB), 0, st, d, nev, d_cnt);
    hipLaunchKernelGGL(k_newton, dim3(std::min(1024, nlinkblk)), dim3(NWB), 0, st, d, nev, d_cnt);
    if (polish) hipLaunchKernelGGL(k_newton_polish, dim3(nlinkblk), dim3(NWB), 0, st, d, nev);
}

// per event: sum, max of the link iteration counts, restarts, unconverged
// and analytic-Jacobian links (out[8 e + 0..4]); one block per 64-link block
// of the root finder, block sums combined with atomics (integers: exact)
__global__ void k_newton_stats_zero(int nev, unsigned long long* __restrict__ acc) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < 5 * nev) acc[t] = 0ull;
}
// kStatBlocks blocks of 256 threads per event stride over its 2S link
// counters; one set of atomics per block (one per 64-link wave made the
// atomics on the five accumulators the cost of the kernel)
constexpr int kStatBlocks = 64;
__global__ __launch_bounds__(256) void k_newton_stats(const EvDesc* __restrict__ evs, int nev,
                                                     unsigned long long* __restrict__ acc) {
    const int e = blockIdx.x / kStatBlocks;
    const int part = blockIdx.x - e * kStatBlocks;
    const EvDesc& ev = evs[e];
    if (!ev.active) return;
    unsigned long long v[5] = {0ull, 0ull, 0ull, 0ull, 0ull};
    for (long long l = (long long)part * 256 + threadIdx.x; l < 2 * ev.S; l += (long long)kStatBlocks * 256) {
        const int x = ev.newton_stat[l];
        const unsigned long long it = (unsigned)(x & 0xFFFFF);
        v[0] += it;
        v[1] = it > v[1] ? it : v[1];
        v[2] += (unsigned)((x >> 20) & 0xFF);
        v[3] += (unsigned)((x >> 28) & 1);
        v[4] += (unsigned)((x >> 29) & 1);
    }
#pragma unroll
    for (int k = 0; k < 5; k++)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const unsigned long long t = __shfl_down(v[k], o, 64);
            v[k] = k == 1 ? (t > v[k] ? t : v[k]) : v[k] + t;
        }
    __shared__ unsigned long long w[4][5];
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < 5; k++) w[wave][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < 4; q++)
#pragma unroll
            for (int k = 0; k < 5; k++) v[k] = k == 1 ? (w[q][k] > v[k] ? w[q][k] : v[k]) : v[k] + w[q][k];
        atomicAdd(&acc[5 * e + 0], v[0]);
        atomicMax(&acc[5 * e + 1], v[1]);
        atomicAdd(&acc[5 * e + 2], v[2]);
        atomicAdd(&acc[5 * e + 3], v[3]);
        atomicAdd(&acc[5 * e + 4], v[4]);
    }
}
__global__ void k_newton_stats_out(int nev, const unsigned long long* __restrict__ acc, double* __restrict__ out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < 5 * nev) out[8 * (t / 5) + t % 5] = (double)acc[t];
}
// d_out holds 16 doubles per event: results in [8e, 8e+5), the integer
// accumulators in the second half [8 nev, 8 nev + 5 nev)
void ipg_launch_newton_stats(const EvDesc* d, int nev, int nlinkblk, double* d_out, hipStream_t st) {
    unsigned long long* acc = reinterpret_cast<unsigned long long*>(d_out + 8 * (size_t)nev);
    const int nb = (5 * nev + 255) / 256;
    hipLaunchKernelGGL(k_newton_stats_zero, dim3(nb), dim3(256), 0, st, nev, acc);
    (void)nlinkblk;
    hipLaunchKernelGGL(k_newton_stats, dim3(kStatBlocks * nev), dim3(256), 0, st, d, nev, acc);
    hipLaunchKernelGGL(k_newton_stats_out, dim3(nb), dim3(256), 0, st, nev, acc, d_out);
}
void ipg_launch_pi_init(const EvDesc* d, int nev, int nblk, hipStream_t st) {
    hipLaunchKernelGGL(k_pi_init, dim3(nblk), dim3(IPG_BLOCK), 0, st, d, nev);
}
void ipg_launch_zero_fields(const EvDesc* d, int nev, int nblk, hipStream_t st) {
    hipLaunchKernelGGL(k_zero_fields, dim3(nblk), dim3(IPG_BLOCK), 0, st, d, nev);
}
void ipg_launch_rho_normals(const EvDesc* d, int nucleus, int k, double* out, hipStream_t st) {
    // single-event helper for parity tests: S sites from the first descriptor
    EvDesc h;
    if (hipMemcpy(&h, d, sizeof(EvDesc), hipMemcpyDeviceToHost) != hipSuccess) return;
    int nb = (int)((h.S + 255) / 256);
    hipLaunchKernelGGL(k_rho_normals, dim3(nb), dim3(256), 0, st, d, nucleus, k, out);
}

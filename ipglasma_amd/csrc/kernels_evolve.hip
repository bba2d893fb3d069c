// kernels_evolve.hip -- classical Yang-Mills leapfrog, T^{mu nu}, Gauss law.
//
// One fused site kernel per leapfrog step replaces the four OpenMP sweeps of
// Evolution::run (Evolution.cpp:405-431):
//   evolvePi  (Evolution.cpp:117-178)  pi += dtau/tau [U phi(+) U^+ + ... - 4 phi]
//   evolveE   (Evolution.cpp:180-293)  E_i += i tau dtau/(2g^2) [plaquettes]_TL
//                                             + i dtau/tau [phi~_i, phi], then TL
//   evolvePhi (Evolution.cpp:90-115)   phi += (tau + dtau/2) dtau pi
//   evolveU   (Evolution.cpp:35-88)    U_i <- (1 + X + X^2/2) U_i,
//                                      X = i g^2 dtau/(tau+dtau/2) E_i
// pi and E depend on the old U and phi only, so the kernel updates pi and E in
// place, then phi and U from the new pi and E, writing phi and U to the other
// half of a ping-pong pair (neighbours still read the old values).  Each site
// reads and writes the six fields once: 1728 algorithmic bytes per site-step
// in the reference's representation (six full 3x3 complex matrices); E1, E2,
// phi and pi are Hermitian and stored as 9 reals, so the kernel moves
// 2 x (2 x 144 + 4 x 72) = 1152 bytes per site-step.
// Neighbours are clamped (Lattice.cpp:19-28).
#include "ipg_device.hpp"
#include "ipg_internal.hpp"

namespace {

struct Nb {
    int s, pX, pY, mX, mY, pXmY, mXpY;
};

__device__ __forceinline__ Nb neighbours(int s, int N) {
    int i = s / N, j = s - (s / N) * N;
    Nb n;
    n.s = s;
    n.pX = clampi(i + 1, N) * N + j;
    n.mX = clampi(i - 1, N) * N + j;
    n.pY = i * N + clampi(j + 1, N);
    n.mY = i * N + clampi(j - 1, N);
    n.pXmY = clampi(i + 1, N) * N + clampi(j - 1, N);
    n.mXpY = clampi(i - 1, N) * N + clampi(j + 1, N);
    return n;
}

// traceless Hermitian part of  E + i c1 A + i c2 B  (E Hermitian, A, B anti-Hermitian)
__device__ __forceinline__ H3 e_update(const H3& E, double c1, const AH& A, double c2, const AH& B) {
    H3 h;
#pragma unroll
    for (int k = 0; k < 3; k++) h.d[k] = E.d[k] - c1 * A.d[k] - c2 * B.d[k];
    const double t = (h.d[0] + h.d[1] + h.d[2]) / 3.0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        h.d[k] -= t;
        h.o[k] = E.o[k] + cd{-c1 * A.o[k].i - c2 * B.o[k].i, c1 * A.o[k].r + c2 * B.o[k].r};
    }
    return h;
}

// What the roles of a site hand each other through LDS: nine doubles a
// matrix, [value][lane] so that a wavefront's accesses are conflict free.
constexpr int kRoleSites = 64;  // sites of a block: one wavefront per role
template <typename X>
__device__ __forceinline__ void x_put(double (*b)[kRoleSites], int lane, const X& a) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
        b[k][lane] = a.d[k];
        b[3 + 2 * k][lane] = a.o[k].r;
        b[4 + 2 * k][lane] = a.o[k].i;
    }
}
template <typename X>
__device__ __forceinline__ X x_get(const double (*b)[kRoleSites], int lane) {
    X a;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        a.d[k] = b[k][lane];
        a.o[k] = cd{b[3 + 2 * k][lane], b[4 + 2 * k][lane]};
    }
    return a;
}

// One step.  A block takes 64 consecutive sites with four wavefronts, each in
// a role of its own (about 460 FP64 multiply-adds a lane each):
//   0  phi~_x, phi~_y and the commutators [phi~_i, phi] of evolveE; pi, phi
//   1  the plaquette U_{1,-2}; E1 and U_x
//   2  the plaquette U_{2,-1}; E2 and U_y
//   3  the plaquette U_12 (U_21 is its conjugate: the two E updates take its
//      anti-Hermitian part with opposite signs) and the x - x^ term of pi
// The stencil is staged in LDS: the sites of the rows i, i+1 and i-1 are
// loaded once (117 planes, all loads of a wavefront in flight together and
// before anything is computed) and the roles read their matrices from there;
// loaded by each role itself the stencil is 333 planes.
//   planes  0 U_x(i), 18 U_y(i), 36 U_y(i+1), 54 U_x(i-1), 72 U_y(i-1),
//          90 phi(i), 99 phi(i+1), 108 phi(i-1)
// A y neighbour is the next lane's value; the two sites past the ends of the
// block are in `ends` (108 values).
constexpr int kSUxI = 0, kSUyI = 18, kSUyP = 36, kSUxM = 54, kSUyM = 72, kSPhI = 90, kSPhP = 99, kSPhM = 108;
constexpr int kStagePlanes = 117;
constexpr int kEUxI = 0, kEUxM = 18, kEPhP = 36;                  // right end: U_x(i), U_x(i-1), phi(i)
constexpr int kELUxI = 45, kELUyI = 63, kELUyP = 81, kELPh = 99;  // left end: U_x(i), U_y(i), U_y(i+1), phi(i)
constexpr int kStageEnds = 108;
typedef double StageRow[kRoleSites];

template <int NP>
__device__ __forceinline__ void stage_planes(StageRow* to, const double* f, size_t S, size_t s, int lane) {
    double v[NP];
    const unsigned ob = lane_offset<false>(s);
#pragma unroll
    for (int k = 0; k < NP; k++) v[k] = gld(f, k * S, ob);
#pragma unroll
    for (int k = 0; k < NP; k++) to[k][lane] = v[k];
}
// matrix at lane q of the stage
__device__ __forceinline__ M3 st_m(const StageRow* f, int q) {
    M3 m;
#pragma unroll
    for (int k = 0; k < 9; k++) m.e[k] = cd{f[2 * k][q], f[2 * k + 1][q]};
    return m;
}
__device__ __forceinline__ H3 st_h(const StageRow* f, int q) {
    H3 h;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        h.d[k] = f[k][q];
        h.o[k] = cd{f[3 + 2 * k][q], f[4 + 2 * k][q]};
    }
    return h;
}
// the same with the value past the block's end taken from `ends`
__device__ __forceinline__ M3 st_me(const StageRow* f, int q, const double* end, bool past) {
    const double* b = past ? end : &f[0][q];
    const int w = past ? 1 : kRoleSites;
    M3 m;
#pragma unroll
    for (int k = 0; k < 9; k++) m.e[k] = cd{b[(2 * k) * w], b[(2 * k + 1) * w]};
    return m;
}
__device__ __forceinline__ H3 st_he(const StageRow* f, int q, const double* end, bool past) {
    const double* b = past ? end : &f[0][q];
    const int w = past ? 1 : kRoleSites;
    H3 h;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        h.d[k] = b[k * w];
        h.o[k] = cd{b[(3 + 2 * k) * w], b[(4 + 2 * k) * w]};
    }
    return h;
}

// One thread per site with everything in registers took 382 of them, one
// wavefront per SIMD, whose chain of loads and products set the pace: 17 us a
// launch at N = 128 (64 blocks of 256 sites left 192 CUs idle), 26 us at
// N = 256, 83 us at N = 512; in roles 7.9, 19.6 and 62.2 us (302 MB of fields
// read and written at N = 512: 4.85 TB/s, a large device copy runs at 4.9; the
// counters read 305 MB in order 0, the neighbour rows come from the L2).
// Also measured: each role loading its own matrices (168 registers, three
// waves per SIMD) 8.7, 20.7, 71 us; at 128 registers it spills (131 us);
// only row i staged 8.0, 21.6, 68 us; blocks that stay and fetch the next
// tile while they store the last 12, 28, 97 us (256 registers and spills).
// order (the tuner's choice; the same results): bit 0: blocks follow each
// other down 64-wide column strips (N a multiple of 64) instead of along the
// rows; bit 1: in the hardware's block order instead of a run of rows per XCD.
// Order 0 is the fastest or level from N = 128 to 768 (58 us at N = 512 against
// 63, 61 and 75 in the tuner's back-to-back launches): there the others fetch
// 31, 31 and 196 MB more, rows that another XCD's L2 holds.
__global__ __launch_bounds__(4 * kRoleSites, 2) void k_step(const EvDesc* __restrict__ evs, int nev, int it, int b0,
                                                            int order) {
    // b0: first block of a launch that covers one event's blocks only (a
    // multiple of 8, so the XCD of a block is unchanged)
    __shared__ StageRow stage[kStagePlanes];
    __shared__ double ends[kStageEnds];
    __shared__ double xch[4][9][kRoleSites];
    constexpr int B4 = IPG_BLOCK / kRoleSites;
    const int bg = (int)blockIdx.x + b0;
    const int e = find_event(evs, nev, bg / B4);
    const EvDesc& ev = evs[e];
    if (!ev.active || it > ev.itmax) return;
    int lb = bg - B4 * ev.block0;
    if (!(order & 2)) lb = xcd_remap(lb, B4 * ev.nblocks);
    const int lane = (int)(threadIdx.x & 63);
    const int role = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int N = ev.N;
    if ((order & 1) && (N & 63) == 0) {
        const int tj = lb / N;
        lb = (lb - tj * N) * (N >> 6) + tj;
    }
    // N is a multiple of 16, S of 256: a block is full or past the end
    if ((long long)lb * kRoleSites >= ev.S) return;
    const size_t s = (size_t)lb * kRoleSites + lane;
    const size_t S = ev.S;
    const int p = (it - 1) & 1;
    const double tau = it * ev.dtau;
    const bool half = it == ev.itmax;
    const double dt = half ? ev.dtau / 2. : ev.dtau;
    const int i = (int)s / N, j = (int)s - i * N;
    const size_t pX = (size_t)min(i + 1, N - 1) * N + j, mX = (size_t)max(i - 1, 0) * N + j;
    const double* __restrict__ Ux = ev.U[p][0];
    const double* __restrict__ Uy = ev.U[p][1];
    const double* __restrict__ phi = ev.phi[p];
    // lane of the y neighbours (clamped), past the block's end or not
    const bool up = j < N - 1, dn = j > 0;
    const int qp = up ? min(lane + 1, 63) : lane, qm = dn ? max(lane - 1, 0) : lane;
    const bool ep = up && lane == 63, em = dn && lane == 0;
    H3 own;
    if (role == 0) {
        own = ldh3(ev.pi, S, s);
        stage_planes<18>(stage + kSUxI, Ux, S, s, lane);
        stage_planes<9>(stage + kSPhI, phi, S, s, lane);
        // right end: the sites of the y neighbour of lane 63 (that lane's own where clamped)
        const int i63 = __builtin_amdgcn_readlane(i, 63), j63 = min(__builtin_amdgcn_readlane(j, 63) + 1, N - 1);
        const size_t r = (size_t)i63 * N + j63, rm = (size_t)max(i63 - 1, 0) * N + j63;
        if (lane < 45) {
            const double* f = lane < 18 ? Ux + lane * S + r : lane < 36 ? Ux + (lane - 18) * S + rm : phi + (lane - 36) * S + r;
            ends[lane] = *f;
        }
    } else if (role == 1) {
        own = ldh3(ev.E1, S, s);
        stage_planes<18>(stage + kSUyI, Uy, S, s, lane);
        stage_planes<9>(stage + kSPhP, phi, S, pX, lane);
        const int i0 = __builtin_amdgcn_readfirstlane(i), jm = max(__builtin_amdgcn_readfirstlane(j) - 1, 0);
        const size_t l = (size_t)i0 * N + jm, lp = (size_t)min(i0 + 1, N - 1) * N + jm;
        if (lane < 63) {
            const double* f = lane < 18   ? Ux + lane * S + l
                              : lane < 36 ? Uy + (lane - 18) * S + l
                              : lane < 54 ? Uy + (lane - 36) * S + lp
                                          : phi + (lane - 54) * S + l;
            ends[kELUxI + lane] = *f;
        }
    } else if (role == 2) {
        own = ldh3(ev.E2, S, s);
        stage_planes<18>(stage + kSUyP, Uy, S, pX, lane);
        stage_planes<9>(stage + kSPhM, phi, S, mX, lane);
    } else {
        stage_planes<18>(stage + kSUxM, Ux, S, mX, lane);
        stage_planes<18>(stage + kSUyM, Uy, S, mX, lane);
    }
    __syncthreads();
    const double a1 = tau * dt / (2. * ev.g * ev.g);
    const double a2 = dt / tau;
    const double cu = ev.g * ev.g * dt / (tau + dt / 2.);
    if (role == 0) {
        const H3 ph = st_h(stage + kSPhI, lane);
        H3 br;
        {
            const M3 u = st_m(stage + kSUxI, lane);
            br = herm_mul(u, mul_hd(st_h(stage + kSPhP, lane), u));  // phi~_x
            x_put(xch[0], lane, commutator(br, ph));
        }
        {
            const M3 u = st_m(stage + kSUyI, lane);
            const H3 t = herm_mul(u, mul_hd(st_he(stage + kSPhI, qp, ends + kEPhP, ep), u));  // phi~_y
            x_put(xch[1], lane, commutator(t, ph));
            br = br + t;
        }
        {
            const M3 u = st_me(stage + kSUyI, qm, ends + kELUyI, em);
            br = br + herm_mul_ad(u, mul_h(st_he(stage + kSPhI, qm, ends + kELPh, em), u));
        }
        __syncthreads();
        br = (br + x_get<H3>(xch[3], lane)) + (-4.) * ph;
        const H3 pin = own + a2 * br;
        sth3(ev.pio, S, s, pin);
        if (!half) sth3(ev.phi[p ^ 1], S, s, ph + ((tau + dt / 2.) * dt) * pin);  // evolvePhi
    } else if (role == 3) {
        {
            const M3 u = st_m(stage + kSUxM, lane);
            x_put(xch[3], lane, herm_mul_ad(u, mul_h(st_h(stage + kSPhM, lane), u)));
        }
        {
            const M3 A = st_m(stage + kSUxI, lane) * st_m(stage + kSUyP, lane);
            x_put(xch[2], lane,
                  ah_mul(A, dag(st_m(stage + kSUyI, lane) * st_me(stage + kSUxI, qp, ends + kEUxI, ep))));
        }
        __syncthreads();
    } else {
        M3 u;
        AH A;
        if (role == 1) {
            u = st_m(stage + kSUxI, lane);
            const M3 l = mul_bd(u, st_me(stage + kSUyP, qm, ends + kELUyP, em));
            A = ah_mul(l, mul_ad(st_me(stage + kSUxI, qm, ends + kELUxI, em), st_me(stage + kSUyI, qm, ends + kELUyI, em)));
        } else {
            u = st_m(stage + kSUyI, lane);
            const M3 l = mul_bd(u, st_me(stage + kSUxM, qp, ends + kEUxM, ep));
            A = ah_mul(l, mul_ad(st_m(stage + kSUyM, lane), st_m(stage + kSUxM, lane)));
        }
        __syncthreads();
        const AH u12 = x_get<AH>(xch[2], lane);
        A = ah_tl(role == 1 ? A + u12 : A - u12);
        const H3 e1 = e_update(own, a1, A, a2, x_get<AH>(xch[role - 1], lane));
        sth3(role == 1 ? ev.E1o : ev.E2o, S, s, e1);
        if (!half) stm(ev.U[p ^ 1][role - 1], S, s, taylor2(cu, e1) * u);  // evolveU
    }
}

// evolvePhi(dtau, 0) and evolveU(dtau, 0) before the loop (Evolution.cpp:393-394)
__global__ __launch_bounds__(IPG_BLOCK) void k_step0(const EvDesc* __restrict__ evs, int nev) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active) return;
    const int lb = xcd_remap(blockIdx.x - ev.block0, ev.nblocks);
    const long long s = (long long)lb * IPG_BLOCK + threadIdx.x;
    if (s >= ev.S) return;
    const size_t S = ev.S;
    const double dt = ev.dtau, tau = 0.;
    M3 ph = ldh(ev.phi[0], S, s) + ((tau + dt / 2.) * dt) * ldh(ev.pi, S, s);
    sth(ev.phi[0], S, s, ph);
    const double cu = ev.g * ev.g * dt / (tau + dt / 2.);
    stm(ev.U[0][0], S, s, taylor2(cu, ldh3(ev.E1, S, s)) * ldm(ev.U[0][0], S, s));
    stm(ev.U[0][1], S, s, taylor2(cu, ldh3(ev.E2, S, s)) * ldm(ev.U[0][1], S, s));
}

// ---- reductions ---------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_down(v, o, 64));
    return v;
}
// deterministic block sum (fixed tree): result valid in thread 0
__device__ double block_sum(double v) {
    __shared__ double w[IPG_BLOCK / 64];
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = 0.;
    if (threadIdx.x == 0)
        for (int k = 0; k < IPG_BLOCK / 64; k++) r += w[k];
    __syncthreads();
    return r;
}
__device__ double block_max(double v) {
    __shared__ double w[IPG_BLOCK / 64];
    v = wave_max(v);
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = 0.;
    if (threadIdx.x == 0)
        for (int k = 0; k < IPG_BLOCK / 64; k++) r = fmax(r, w[k]);
    __syncthreads();
    return r;
}

// ---- T^{mu nu} (Evolution.cpp:659-1246) ---------------------------------------
__device__ __forceinline__ M3 m4(const M3& a, const M3& b, const M3& c, const M3& d) { return ((a * b) * c) * d; }
__device__ __forceinline__ M3 m3(const M3& a, const M3& b, const M3& c) { return (a * b) * c; }
// ((P1-P2) - tr/3) + P3 - P4 - tr(P3-P4)/3
__device__ __forceinline__ M3 tlquad(const M3& P1, const M3& P2, const M3& P3, const M3& P4) {
    return traceless(P1 - P2) + traceless(P3 - P4);
}

// Each block below reloads its inputs (L1/L2 hits) after a compiler memory
// barrier, so that only the matrices of one term are live at a time.
#define IPG_FENCE() asm volatile("" ::: "memory")

// T^{mu nu} in three passes (register pressure): diagonal components,
// T^{tau eta} and T^{xy}; the block sums of T^tautau
__global__ __launch_bounds__(IPG_BLOCK) void k_tmunu_a(const EvDesc* __restrict__ evs, int nev, int it) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active || it != ev.itmax) return;
    const int lb = xcd_remap(blockIdx.x - ev.block0, ev.nblocks);
    const long long s = (long long)lb * IPG_BLOCK + threadIdx.x;
    double ttsum = 0.;
    if (s < ev.S) {
        const size_t S = ev.S;
        const int N = ev.N;
        const int p = (it - 1) & 1;
        const double* Ux = ev.U[p][0];
        const double* Uy = ev.U[p][1];
        const double* phi = ev.phi[p];
        const double* E1 = ev.E1;
        const double* E2 = ev.E2;
        [[maybe_unused]] const double* PI = ev.pi;
        [[maybe_unused]] const double tau = it * ev.dtau, g = ev.g, a = ev.a;
        const int i = (int)(s / N), j = (int)(s - (s / N) * N);
        auto at = [&](int di, int dj) { return (size_t)clampi(i + di, N) * N + clampi(j + dj, N); };
        // the neighbours of the whole T^{mu nu} stencil (each pass uses a subset)
        [[maybe_unused]] const size_t pX = at(1, 0), pY = at(0, 1), pXY = at(1, 1), mX = at(-1, 0), mY = at(0, -1);
        [[maybe_unused]] const size_t mXpY = at(-1, 1), pXmY = at(1, -1), p2X = at(2, 0), p2Y = at(0, 2);
        [[maybe_unused]] const size_t p2XY = at(2, 1), pX2Y = at(1, 2);
        double* T = ev.T;
        [[maybe_unused]] const double a2 = a * a, a4 = a2 * a2, a5 = a4 * a, a6 = a4 * a2;
        // phi gradients: gX = Ux phi(x+x) Ux^+ - phi, gY, gXY1 = Ux(+y) phi(+x+y) Ux(+y)^+ - phi(+y),
        // gXY2 = Uy(+x) phi(+x+y) Uy(+x)^+ - phi(+x)
        auto gX = [&]() { M3 u = ldm<true>(Ux, S, s); return m3(u, ldh<true>(phi, S, pX), dag(u)) - ldh<true>(phi, S, s); };
        auto gY = [&]() { M3 u = ldm<true>(Uy, S, s); return m3(u, ldh<true>(phi, S, pY), dag(u)) - ldh<true>(phi, S, s); };
        auto gXY1 = [&]() { M3 u = ldm<true>(Ux, S, pY); return m3(u, ldh<true>(phi, S, pXY), dag(u)) - ldh<true>(phi, S, pY); };
        auto gXY2 = [&]() { M3 u = ldm<true>(Uy, S, pX); return m3(u, ldh<true>(phi, S, pXY), dag(u)) - ldh<true>(phi, S, pX); };

        // electric and longitudinal (Evolution.cpp:754-814)
        double tt, xx, yy, ee;
        {
            const M3 e1 = ldh<true>(E1, S, s), e1p = ldh<true>(E1, S, pY), e2 = ldh<true>(E2, S, s), e2p = ldh<true>(E2, S, pX);
            const double t11 = retrprod(e1, e1), t1p = retrprod(e1p, e1p), t22 = retrprod(e2, e2),
                         t2p = retrprod(e2p, e2p);
            double lng = 0.;
            {
                M3 q = ldh<true>(PI, S, s);
                lng += retrprod(q, q);
                q = ldh<true>(PI, S, pX);
                lng += retrprod(q, q);
                q = ldh<true>(PI, S, pY);
                lng += retrprod(q, q);
                q = ldh<true>(PI, S, pXY);
                lng += retrprod(q, q);
                lng /= 4.;
            }
            const double gt = g * g / tau / tau;
            tt = gt * (t11 + t1p + t22 + t2p) / 2. + lng;
            xx = gt * (-t11 - t1p + t22 + t2p) / 2. + lng;
            yy = gt * (t11 + t1p - t22 - t2p) / 2. + lng;
            ee = 1. / tau / tau * (gt * (t11 + t1p + t22 + t2p) / 2. - lng);
        }
        IPG_FENCE();
        // magnetic and transverse phi gradients (Evolution.cpp:816-905)
        {
            double rplaq = 3.0;
            if (i != N - 1) {
                const M3 ux = ldm<true>(Ux, S, s);
                rplaq = retrprod(ux, ldm<true>(Uy, S, pX) * mul_bd(dag(ldm<true>(Ux, S, pY)), ldm<true>(Uy, S, s)));
            }
            double A, B, C, D;
            {
                M3 q = gX();
                A = retrprod(q, q);
            }
            {
                M3 q = gXY1();
                B = retrprod(q, q);
            }
            {
                M3 q = gY();
                C = retrprod(q, q);
            }
            {
                M3 q = gXY2();
                D = retrprod(q, q);
            }
            const double mag = 2. / (g * g) * (3.0 - rplaq);
            const double h = 0.5 / tau / tau;
            tt = (tt + mag) + h * (A + B + C + D);
            xx = (xx + mag) + h * (A + B - C - D);
            yy = (yy + mag) + h * (-A - B + C + D);
            ee = ee + 1. / tau / tau * (-mag + h * (A + B + C + D));
        }
        T[0 * S + s] = tt / a4;
        T[1 * S + s] = xx / a4;
        T[2 * S + s] = yy / a4;
        T[3 * S + s] = ee / a6;
        ttsum = tt / a4;
        IPG_FENCE();
        // T^{tau eta}
        {
            double re = retrprod(ldh<true>(E1, S, s), gX());
            re += retrprod(ldh<true>(E1, S, pY), gXY1());
            re += retrprod(ldh<true>(E2, S, s), gY());
            re += retrprod(ldh<true>(E2, S, pX), gXY2());
            T[6 * S + s] = (g / tau / tau / tau * re) / a5;
        }
        IPG_FENCE();
        // T^{xy}
        {
            const M3 ux = ldm<true>(Ux, S, s), uy = ldm<true>(Uy, S, s);
            double b;
            {
                const M3 el = (-1. / 4. * g * g * (ldh<true>(E1, S, s) + m3(uy, ldh<true>(E1, S, pY), dag(uy)))) *
                              (ldh<true>(E2, S, s) + m3(ux, ldh<true>(E2, S, pX), dag(ux)));
                b = 4. * tr(el).r;
            }
            const M3 yl = m3(uy, gXY1(), dag(uy));  // U_y gXY1 U_y^+
            const M3 xl = m3(ux, gXY2(), dag(ux));  // U_x gXY2 U_x^+
            const M3 gx = gX(), gy = gY();
            b += retrprod(gx, gy) + retrprod(yl, gy) + retrprod(gx, xl) + retrprod(yl, xl);
            T[7 * S + s] = (2. / tau / tau * (0.25 * b)) / a4;
        }
        IPG_FENCE();
    }
    double bs = block_sum(ttsum);
    if (threadIdx.x == 0) ev.partial[lb] = bs;
}

// clover parts of T^{tau x}, T^{tau y}, T^{x eta}, T^{y eta}
__global__ __launch_bounds__(IPG_BLOCK) void k_tmunu_b(const EvDesc* __restrict__ evs, int nev, int it) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active || it != ev.itmax) return;
    const int lb = xcd_remap(blockIdx.x - ev.block0, ev.nblocks);
    const long long s = (long long)lb * IPG_BLOCK + threadIdx.x;
    if (s < ev.S) {
        const size_t S = ev.S;
        const int N = ev.N;
        const int p = (it - 1) & 1;
        const double* Ux = ev.U[p][0];
        const double* Uy = ev.U[p][1];
        const double* phi = ev.phi[p];
        const double* E1 = ev.E1;
        const double* E2 = ev.E2;
        [[maybe_unused]] const double* PI = ev.pi;
        [[maybe_unused]] const double tau = it * ev.dtau, g = ev.g, a = ev.a;
        const int i = (int)(s / N), j = (int)(s - (s / N) * N);
        auto at = [&](int di, int dj) { return (size_t)clampi(i + di, N) * N + clampi(j + dj, N); };
        // the neighbours of the whole T^{mu nu} stencil (each pass uses a subset)
        [[maybe_unused]] const size_t pX = at(1, 0), pY = at(0, 1), pXY = at(1, 1), mX = at(-1, 0), mY = at(0, -1);
        [[maybe_unused]] const size_t mXpY = at(-1, 1), pXmY = at(1, -1), p2X = at(2, 0), p2Y = at(0, 2);
        [[maybe_unused]] const size_t p2XY = at(2, 1), pX2Y = at(1, 2);
        double* T = ev.T;
        [[maybe_unused]] const double a2 = a * a, a4 = a2 * a2, a5 = a4 * a, a6 = a4 * a2;
        // phi gradients: gX = Ux phi(x+x) Ux^+ - phi, gY, gXY1 = Ux(+y) phi(+x+y) Ux(+y)^+ - phi(+y),
        // gXY2 = Uy(+x) phi(+x+y) Uy(+x)^+ - phi(+x)
        auto gX = [&]() { M3 u = ldm<true>(Ux, S, s); return m3(u, ldh<true>(phi, S, pX), dag(u)) - ldh<true>(phi, S, s); };
        auto gY = [&]() { M3 u = ldm<true>(Uy, S, s); return m3(u, ldh<true>(phi, S, pY), dag(u)) - ldh<true>(phi, S, s); };
        auto gXY1 = [&]() { M3 u = ldm<true>(Ux, S, pY); return m3(u, ldh<true>(phi, S, pXY), dag(u)) - ldh<true>(phi, S, pY); };
        auto gXY2 = [&]() { M3 u = ldm<true>(Uy, S, pX); return m3(u, ldh<true>(phi, S, pXY), dag(u)) - ldh<true>(phi, S, pX); };

        // T^{tau x}, T^{x eta}, T^{tau y}, T^{y eta} (Evolution.cpp:1047-1234).
        // The clover combinations enter with opposite signs, e.g. the T^{x eta}
        // clover (Pb - Pa)_TL + (Pd - Pc)_TL is -X1.
        double ttx_im, tty_im, xe_im, ye_im;
        {
            // X1 = (Pa - Pb)_TL + (Pc - Pd)_TL,
            // Pa = Uy Ux(+y) Uy(+x)^+ Ux^+, Pb = Ux Uy(+x) Ux(+y)^+ Uy^+
            const M3 ux = ldm<true>(Ux, S, s), uy = ldm<true>(Uy, S, s);
            M3 X = traceless(m4(uy, ldm<true>(Ux, S, pY), dag(ldm<true>(Uy, S, pX)), dag(ux)) -
                             m4(ux, ldm<true>(Uy, S, pX), dag(ldm<true>(Ux, S, pY)), dag(uy)));
            {
                const M3 UxmX = ldm<true>(Ux, S, mX), UxmXpY = ldm<true>(Ux, S, mXpY), UymX = ldm<true>(Uy, S, mX);
                X = X + traceless(m4(dag(UxmX), UymX, UxmXpY, dag(uy)) - m4(uy, dag(UxmXpY), dag(UymX), UxmX));
            }
            ttx_im = imtrprod(ldh<true>(E2, S, s), X);
            xe_im = -imtrprod(X, gY());
        }
        IPG_FENCE();
        {
            // Y1 = (Pb - Pa)_TL + (Qc - Qd)_TL
            const M3 ux = ldm<true>(Ux, S, s), uy = ldm<true>(Uy, S, s);
            M3 Y = traceless(m4(ux, ldm<true>(Uy, S, pX), dag(ldm<true>(Ux, S, pY)), dag(uy)) -
                             m4(uy, ldm<true>(Ux, S, pY), dag(ldm<true>(Uy, S, pX)), dag(ux)));
            {
                const M3 UymY = ldm<true>(Uy, S, mY), UxmY = ldm<true>(Ux, S, mY), UypXmY = ldm<true>(Uy, S, pXmY);
                Y = Y + traceless(m4(dag(UymY), UxmY, UypXmY, dag(ux)) - m4(ux, dag(UypXmY), dag(UxmY), UymY));
            }
            tty_im = imtrprod(ldh<true>(E1, S, s), Y);
            ye_im = -imtrprod(Y, gX());
        }
        IPG_FENCE();
        {
            // X2 = (Pe - Pf)_TL + (Pg - Ph)_TL
            const M3 UxpX = ldm<true>(Ux, S, pX), UxpXpY = ldm<true>(Ux, S, pXY), Uyp2X = ldm<true>(Uy, S, p2X);
            const M3 UypX = ldm<true>(Uy, S, pX);
            M3 X = traceless(m4(UypX, UxpXpY, dag(Uyp2X), dag(UxpX)) - m4(UxpX, Uyp2X, dag(UxpXpY), dag(UypX)));
            {
                const M3 ux = ldm<true>(Ux, S, s), uy = ldm<true>(Uy, S, s), UxpY = ldm<true>(Ux, S, pY);
                X = X + traceless(m4(dag(ux), uy, UxpY, dag(UypX)) - m4(UypX, dag(UxpY), dag(uy), ux));
            }
            ttx_im += imtrprod(ldh<true>(E2, S, pX), X);
            xe_im -= imtrprod(X, gXY2());
        }
        IPG_FENCE();
        {
            // Y2 = (Qe - Qf)_TL + (Qg - Qh)_TL
            const M3 UxpY = ldm<true>(Ux, S, pY), UypXpY = ldm<true>(Uy, S, pXY), Uxp2Y = ldm<true>(Ux, S, p2Y);
            const M3 UypY = ldm<true>(Uy, S, pY);
            M3 Y = traceless(m4(UxpY, UypXpY, dag(Uxp2Y), dag(UypY)) - m4(UypY, Uxp2Y, dag(UypXpY), dag(UxpY)));
            {
                const M3 ux = ldm<true>(Ux, S, s), uy = ldm<true>(Uy, S, s), UypX = ldm<true>(Uy, S, pX);
                Y = Y + traceless(m4(dag(uy), ux, UypX, dag(UxpY)) - m4(UxpY, dag(UypX), dag(ux), uy));
            }
            tty_im += imtrprod(ldh<true>(E1, S, pY), Y);
            ye_im -= imtrprod(Y, gXY1());
        }
        // raw clover sums, finished by k_tmunu_c
        T[4 * S + s] = ttx_im;
        T[5 * S + s] = tty_im;
        T[8 * S + s] = xe_im;
        T[9 * S + s] = ye_im;
    }
}

// pi grad-phi and E pi parts; finishes the four flux components
__global__ __launch_bounds__(IPG_BLOCK) void k_tmunu_c(const EvDesc* __restrict__ evs, int nev, int it) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active || it != ev.itmax) return;
    const int lb = xcd_remap(blockIdx.x - ev.block0, ev.nblocks);
    const long long s = (long long)lb * IPG_BLOCK + threadIdx.x;
    if (s < ev.S) {
        const size_t S = ev.S;
        const int N = ev.N;
        const int p = (it - 1) & 1;
        const double* Ux = ev.U[p][0];
        const double* Uy = ev.U[p][1];
        const double* phi = ev.phi[p];
        const double* E1 = ev.E1;
        const double* E2 = ev.E2;
        [[maybe_unused]] const double* PI = ev.pi;
        [[maybe_unused]] const double tau = it * ev.dtau, g = ev.g, a = ev.a;
        const int i = (int)(s / N), j = (int)(s - (s / N) * N);
        auto at = [&](int di, int dj) { return (size_t)clampi(i + di, N) * N + clampi(j + dj, N); };
        // the neighbours of the whole T^{mu nu} stencil (each pass uses a subset)
        [[maybe_unused]] const size_t pX = at(1, 0), pY = at(0, 1), pXY = at(1, 1), mX = at(-1, 0), mY = at(0, -1);
        [[maybe_unused]] const size_t mXpY = at(-1, 1), pXmY = at(1, -1), p2X = at(2, 0), p2Y = at(0, 2);
        [[maybe_unused]] const size_t p2XY = at(2, 1), pX2Y = at(1, 2);
        double* T = ev.T;
        [[maybe_unused]] const double a2 = a * a, a4 = a2 * a2, a5 = a4 * a, a6 = a4 * a2;
        // pi phi-gradient parts of T^{tau x} and T^{tau y}
        double ttx_re, tty_re;
        const double ttx_im = T[4 * S + s], tty_im = T[5 * S + s], xe_im = T[8 * S + s], ye_im = T[9 * S + s];
        IPG_FENCE();
        {
            M3 u = ldm<true>(Ux, S, s), v = ldm<true>(Ux, S, mX);
            ttx_re = retrprod(ldh<true>(PI, S, s), m3(u, ldh<true>(phi, S, pX), dag(u)) - m3(dag(v), ldh<true>(phi, S, mX), v));
            u = ldm<true>(Ux, S, pY);
            v = ldm<true>(Ux, S, mXpY);
            ttx_re += retrprod(ldh<true>(PI, S, pY), m3(u, ldh<true>(phi, S, pXY), dag(u)) - m3(dag(v), ldh<true>(phi, S, mXpY), v));
            u = ldm<true>(Ux, S, pX);
            v = ldm<true>(Ux, S, s);
            ttx_re += retrprod(ldh<true>(PI, S, pX), m3(u, ldh<true>(phi, S, p2X), dag(u)) - m3(dag(v), ldh<true>(phi, S, s), v));
            u = ldm<true>(Ux, S, pXY);
            v = ldm<true>(Ux, S, pY);
            ttx_re += retrprod(ldh<true>(PI, S, pXY), m3(u, ldh<true>(phi, S, p2XY), dag(u)) - m3(dag(v), ldh<true>(phi, S, pY), v));
        }
        IPG_FENCE();
        {
            M3 u = ldm<true>(Uy, S, s), v = ldm<true>(Uy, S, mY);
            tty_re = retrprod(ldh<true>(PI, S, s), m3(u, ldh<true>(phi, S, pY), dag(u)) - m3(dag(v), ldh<true>(phi, S, mY), v));
            u = ldm<true>(Uy, S, pX);
            v = ldm<true>(Uy, S, pXmY);
            tty_re += retrprod(ldh<true>(PI, S, pX), m3(u, ldh<true>(phi, S, pXY), dag(u)) - m3(dag(v), ldh<true>(phi, S, pXmY), v));
            u = ldm<true>(Uy, S, pY);
            v = ldm<true>(Uy, S, s);
            tty_re += retrprod(ldh<true>(PI, S, pY), m3(u, ldh<true>(phi, S, p2Y), dag(u)) - m3(dag(v), ldh<true>(phi, S, s), v));
            u = ldm<true>(Uy, S, pXY);
            v = ldm<true>(Uy, S, pX);
            tty_re += retrprod(ldh<true>(PI, S, pXY), m3(u, ldh<true>(phi, S, pX2Y), dag(u)) - m3(dag(v), ldh<true>(phi, S, pX), v));
        }
        T[4 * S + s] = (2. / tau / 8. * ttx_im - 2. / 8. / tau * ttx_re) / a4;
        T[5 * S + s] = (2. / tau / 8. * tty_im - 2. / 8. / tau * tty_re) / a4;
        IPG_FENCE();
        // E pi parts of T^{x eta}, T^{y eta}
        {
            M3 u = ldm<true>(Ux, S, s);
            double r1 = retrprod(ldh<true>(E1, S, s), ldh<true>(PI, S, s) + m3(u, ldh<true>(PI, S, pX), dag(u)));
            u = ldm<true>(Ux, S, pY);
            r1 += retrprod(ldh<true>(E1, S, pY), ldh<true>(PI, S, pY) + m3(u, ldh<true>(PI, S, pXY), dag(u)));
            T[8 * S + s] = (-2. / tau / tau * (1. / 4. * g * r1 + 1. / 8. / g * xe_im)) / a5;
        }
        IPG_FENCE();
        {
            M3 u = ldm<true>(Uy, S, s);
            double r1 = retrprod(ldh<true>(E2, S, s), ldh<true>(PI, S, s) + m3(u, ldh<true>(PI, S, pY), dag(u)));
            u = ldm<true>(Uy, S, pX);
            r1 += retrprod(ldh<true>(E2, S, pX), ldh<true>(PI, S, pX) + m3(u, ldh<true>(PI, S, pXY), dag(u)));
            T[9 * S + s] = (-2. / tau / tau * (1. / 4. * g * r1 + 1. / 8. / g * ye_im)) / a5;
        }
    }
}

__global__ __launch_bounds__(IPG_BLOCK) void k_gauss(const EvDesc* __restrict__ evs, int nev, int it) {
    const int e = find_event(evs, nev, blockIdx.x);
    const EvDesc& ev = evs[e];
    if (!ev.active || it != ev.itmax) return;
    const int lb = xcd_remap(blockIdx.x - ev.block0, ev.nblocks);
    const long long s = (long long)lb * IPG_BLOCK + threadIdx.x;
    double v = 0.;
    if (s < ev.S) {
        const size_t S = ev.S;
        const int p = (it - 1) & 1;
        const Nb n = neighbours((int)s, ev.N);
        const M3 uxm = ldm(ev.U[p][0], S, n.mX), uym = ldm(ev.U[p][1], S, n.mY);
        const M3 ph = ldh(ev.phi[p], S, s), pp = ldh(ev.pi, S, s);
        M3 G = mul_ad(uxm, ldh(ev.E1, S, n.mX)) * uxm - ldh(ev.E1, S, s);
        G = G + mul_ad(uym, ldh(ev.E2, S, n.mY)) * uym - ldh(ev.E2, S, s);
        G = G - mul_i(1.0, ph * pp - pp * ph);
        v = square(G);
    }
    double bm = block_max(v);
    if (threadIdx.x == 0) ev.partial[ev.nblocks + lb] = bm;
}

// per event: out[4e+0] = sum T^tautau (fm^-4), out[4e+1] = Gauss max
__global__ __launch_bounds__(IPG_BLOCK) void k_finish(const EvDesc* __restrict__ evs, int nev, int it,
                                                     double* __restrict__ out) {
    const int e = blockIdx.x;
    if (e >= nev) return;
    const EvDesc& ev = evs[e];
    if (!ev.active || it != ev.itmax) return;
    const int nb = (int)((ev.S + IPG_BLOCK - 1) / IPG_BLOCK);
    // fixed-order per-thread partial sums, then a fixed tree
    double sm = 0., mx = 0.;
    for (int b = threadIdx.x; b < ev.nblocks; b += IPG_BLOCK) {
        int l = b;  // logical block index
        if (l < nb) {
            sm += ev.partial[l];
            mx = fmax(mx, ev.partial[ev.nblocks + l]);
        }
    }
    double ts = block_sum(sm);
    double tm = block_max(mx);
    if (threadIdx.x == 0) {
        out[4 * e + 0] = ts;
        out[4 * e + 1] = tm;
    }
}

}  // namespace

void ipg_launch_step0(const EvDesc* d_evs, int nev, int nblk, hipStream_t st) {
    hipLaunchKernelGGL(k_step0, dim3(nblk), dim3(IPG_BLOCK), 0, st, d_evs, nev);
}
void ipg_launch_step(const EvDesc* d_evs, int nev, int nblk, int it, hipStream_t st, int variant) {
    ipg_launch_step_event(d_evs, nev, 0, nblk, it, st, variant);
}
// block0, nblocks: in blocks of IPG_BLOCK sites, as everywhere else
void ipg_launch_step_event(const EvDesc* d_evs, int nev, int block0, int nblocks, int it, hipStream_t st,
                           int variant) {
    constexpr int B4 = IPG_BLOCK / kRoleSites;
    hipLaunchKernelGGL(k_step, dim3(B4 * nblocks), dim3(4 * kRoleSites), 0, st, d_evs, nev, it, B4 * block0, variant);
}
void ipg_launch_tmunu(const EvDesc* d_evs, int nev, int nblk, int it, hipStream_t st) {
    hipLaunchKernelGGL(k_tmunu_a, dim3(nblk), dim3(IPG_BLOCK), 0, st, d_evs, nev, it);
    hipLaunchKernelGGL(k_tmunu_b, dim3(nblk), dim3(IPG_BLOCK), 0, st, d_evs, nev, it);
    hipLaunchKernelGGL(k_tmunu_c, dim3(nblk), dim3(IPG_BLOCK), 0, st, d_evs, nev, it);
}
void ipg_launch_gauss(const EvDesc* d_evs, int nev, int nblk, int it, hipStream_t st) {
    hipLaunchKernelGGL(k_gauss, dim3(nblk), dim3(IPG_BLOCK), 0, st, d_evs, nev, it);
}
void ipg_launch_finish(const EvDesc* d_evs, int nev, int it, double* d_out, hipStream_t st) {
    hipLaunchKernelGGL(k_finish, dim3(nev), dim3(IPG_BLOCK), 0, st, d_evs, nev, it, d_out);
}

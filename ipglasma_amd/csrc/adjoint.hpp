// adjoint.hpp -- reverse mode of one leapfrog step and of T^tautau at one
// site (Evolution.cpp:35-293 and 754-905), host+device.
//
// Convention: for a real loss L and a complex matrix Z the cotangent is
// Zb = dL/dRe Z + i dL/dIm Z, so that dL = Re tr(Zb^+ dZ).  Rules used:
//   Y = A B      ->  Ab += Yb B^+,  Bb += A^+ Yb
//   Y = A^+      ->  Ab += Yb^+
//   Y = c A      ->  Ab += conj(c) Yb
//   Y = TL(A)    ->  Ab += TL(Yb)              (traceless part: self-adjoint)
//   y = Re tr(Z Z) -> Zb += 2 yb Z^+
// Links are general complex matrices (the second-order update is not
// unitary); E, phi and pi are Hermitian, and their cotangents are projected
// on the Hermitian matrices where they are stored.
//
// Forward step at tau (lattice units), the reference's order:
//   pi'  = pi + (dtau/tau) [Ux phi(x+x) Ux^+ + Ux(x-x)^+ phi(x-x) Ux(x-x)
//                           + (same in y) - 4 phi]
//   E1'  = TL(E1 + c1 TL(U12 + U1m2 - h.c.) + c2 [Ux phi(x+x) Ux^+, phi])
//   E2'  = TL(E2 + c1 TL(U12^+ + U2m1 - h.c.) + c2 [Uy phi(x+y) Uy^+, phi])
//   phi' = phi + (tau + dtau/2) dtau pi'
//   U'   = (1 + X + X^2/2) U,  X = i g^2 dtau / (tau + dtau/2) E'
// with c1 = i tau dtau / (2 g^2), c2 = i dtau / tau.
#pragma once
#include "su3.hpp"

namespace ipgad {

IPG_HD M3 hproj(const M3& z) { return 0.5 * (z + dag(z)); }
IPG_HD M3 cscale(cd c, const M3& a) {
    M3 r;
#pragma unroll
    for (int k = 0; k < 9; k++) r.e[k] = c * a.e[k];
    return r;
}

// Y = A F A^+ (F Hermitian):  Ab += (Yb + Yb^+) A F,  Fb += A^+ Yb A
IPG_HD void adj_conj(const M3& A, const M3& F, const M3& Yb, M3& Ab, M3& Fb) {
    Ab = Ab + (Yb + dag(Yb)) * (A * F);
    Fb = Fb + mul_ad(A, Yb) * A;
}
// Y = V^+ G V (G Hermitian):  Vb += G V (Yb + Yb^+),  Gb += V Yb V^+
IPG_HD void adj_conjd(const M3& V, const M3& G, const M3& Yb, M3& Vb, M3& Gb) {
    Vb = Vb + (G * V) * (Yb + dag(Yb));
    Gb = Gb + mul_bd(V * Yb, V);
}
// Y = M1 M2 M3 M4: cotangents of the four factors (each product is formed
// just before its last use)
IPG_HD void adj_prod4(const M3& M1, const M3& M2, const M3& M3_, const M3& M4, const M3& Yb, M3& B1, M3& B2,
                      M3& B3, M3& B4) {
    const M3 P34 = M3_ * M4;
    B1 = mul_bd(Yb, M2 * P34);               // Yb (M2 M3 M4)^+
    B2 = mul_bd(mul_ad(M1, Yb), P34);        // M1^+ Yb (M3 M4)^+
    const M3 P12 = M1 * M2;
    B3 = mul_bd(mul_ad(P12, Yb), M4);        // (M1 M2)^+ Yb M4^+
    B4 = mul_ad(P12 * M3_, Yb);              // (M1 M2 M3)^+ Yb
}

// ---- link update U' = (1 + X + X^2/2) U, X = i kappa E' ---------------------------
IPG_HD M3 taylor_m(const M3& X) { return m_one() + X * (m_one() + 0.5 * X); }
IPG_HD M3 u_fwd(const M3& U, const M3& E, double kappa) { return taylor_m(cscale(cd{0., kappa}, E)) * U; }
// Ub += M^+ Yb,  Eb += -i kappa (Mb + (Mb X^+ + X^+ Mb)/2),  Mb = Yb U^+
IPG_HD void u_adj(const M3& U, const M3& E, double kappa, const M3& Yb, M3& Ub, M3& Eb) {
    const M3 X = cscale(cd{0., kappa}, E);
    const M3 M = taylor_m(X);
    Ub = Ub + mul_ad(M, Yb);
    const M3 Mb = mul_bd(Yb, U);
    const M3 Xd = dag(X);
    const M3 Xb = Mb + 0.5 * (Mb * Xd + Xd * Mb);
    Eb = Eb + cscale(cd{0., -kappa}, Xb);
}

// ---- the leapfrog step in reverse, gathered per site -------------------------------
// The cotangents a site's own fields receive, from the sites of its stencil
// (the host test holds the same sums scattered site by site).  Z1, Z2 are the traceless
// Hermitian cotangents of E1', E2' and bb = (dtau/tau) of pi''s.  With
// a = tau dtau / (2 g^2), the plaquettes of E' have the cotangents
//   U12 = Ux Uy(+x) Ux(+y)^+ Uy^+             -2ia (Z1 - Z2)
//   U1m2 = Ux Uy(+x-y)^+ Ux(-y)^+ Uy(-y)      -2ia Z1
//   U2m1 = Uy Ux(-x+y)^+ Uy(-x)^+ Ux(-x)      -2ia Z2
// and a link U_x(t) enters three of each through the loop above it (corners t,
// t+x, t+y) and three through the loop below it (corners t-y, t+x-y, t).  The
// lattice is clamped: at its edges a site is its own neighbour, so some
// sources are missing and others come twice (the weights and extra terms).
// The y link is the x link with the axes exchanged (x <-> y, Z1 <-> Z2), so
// one code serves both: F has the site's coordinates p along and q across the
// link, N, and uf, uo (links along and across), zf, zo, ph, bb at the clamped
// offset (dp, dq) from it.

// keeps the scheduler from having every factor of a sum loaded at once
IPG_HD void adj_fence() {
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_sched_barrier(0);
#endif
}
// the loop above the link, in units of -2ia.  First the sources every site has
// (weights 0 where an edge takes one away), then, on the edges, the sources
// that are there twice: the same body with other sites and weights, so that
// the code stays small (the instruction cache holds 64 KB).
template <class F>
IPG_HD M3 adj_link_above(const F& f) {
    const int N = f.N;
    M3 r = m_zero();
#pragma unroll 1
    for (int rep = 0; rep < 3; rep++) {
        // 1: the site is its own neighbour below (U1m2 of the site itself), 2:
        // its own neighbour behind (U2m1 of the site itself)
        if ((rep == 1 && f.q != 0) || (rep == 2 && f.p != 0)) continue;
        const int l = rep == 1 ? 0 : 1, m = rep == 2 ? 0 : 1;
        const double wd = rep == 0 ? 1. : 0., wz = rep == 1 || (rep == 0 && f.q < N - 1) ? 1. : 0.;
        const double wo = rep == 2 || (rep == 0 && f.p < N - 1) ? 1. : 0.;
        const M3 G = mul_bd(f.uf(0, l), f.uo(m, 0));
        const M3 U = f.uo(0, 0);
        const M3 T = mac_mh(mul_h(wd * (f.zf(0, 0) - f.zo(0, 0)), U), U, -wz * f.zf(0, l));
        r = mac(r, T, G);
        adj_fence();
        r = mac(r, U, mul_mh(G, wo * f.zo(m, 0)));
        adj_fence();
    }
    return r;
}
// the loop below the link, in units of -2ia
template <class F>
IPG_HD M3 adj_link_below(const F& f) {
    const int N = f.N;
    M3 r = m_zero();
#pragma unroll 1
    for (int rep = 0; rep < 2; rep++) {
        // 1: the site is its own neighbour above (U12 and U2m1 of its own row)
        if (rep == 1 && f.q != N - 1) continue;
        const int l = rep == 0 ? -1 : 0;
        const double wc = rep == 0 ? 1. : 0., wb = rep == 1 || f.q > 0 ? 1. : 0., we = f.p < N - 1 ? wb : 0.;
        const M3 U = f.uo(0, l), u = f.uf(0, l);
        // Z U^+ - U^+ D = (U Z - D U)^+
        const M3 T = mac_mh(mul_h(-wb * (f.zf(0, l) - f.zo(0, l)), U), U, wc * f.zf(0, 0));
        const M3 X = mac_ad(mul_ad(T, u), U, mul_mh(u, -we * f.zo(1, l)));
        r = mac(r, X, f.uo(1, l));
        adj_fence();
        if (f.p == 0 && wb != 0.) {
            const M3 V = f.uo(0, l);
            r = r - mul_ad(V, f.uf(0, l)) * mul_h(f.zo(0, l), V);
        }
        adj_fence();
    }
    return r;
}
// bb of the sites whose neighbour against the link's direction is this one
template <class F>
IPG_HD H3 adj_bb_sum(const F& f) {
    const double w1 = f.p < f.N - 1 ? 1. : 0., w0 = f.p == 0 ? 1. : 0.;
    return w1 * f.bb(1, 0) + w0 * f.bb(0, 0);
}
// bb + the cotangent of phi~ from the commutator of E', k = dtau/tau
template <class F>
IPG_HD H3 adj_q(const F& f, int dp, double k) {
    return f.bb(dp, 0) + herm_mi(k, commutator(f.zf(dp, 0), f.ph(dp, 0)));
}
// the link's share of the commutator of E' and of the pi' stencil
template <class F>
IPG_HD M3 adj_link_phi(const F& f, double k) {
    const M3 u = f.uf(0, 0);
    const M3 a = mul_mh(mul_h(adj_q(f, 0, k), u), f.ph(1, 0));
    adj_fence();
    return 2. * (a + mul_h(f.ph(0, 0), mul_mh(u, adj_bb_sum(f))));
}
// phi's share through the links of this direction (without -4 bb)
template <class F>
IPG_HD H3 adj_phi_dir(const F& f, double k) {
    const M3 u = f.uf(0, 0);
    const H3 tx = herm_mul(u, mul_hd(f.ph(1, 0), u));
    H3 r = herm_mi(k, commutator(tx, f.zf(0, 0))) + herm_mul(u, mul_hd(adj_bb_sum(f), u));
    adj_fence();
    if (f.p > 0) {
        const M3 v = f.uf(-1, 0);
        r = r + herm_mul_ad(v, mul_h(adj_q(f, -1, k), v));
    }
    if (f.p == f.N - 1) r = r + herm_mul_ad(u, mul_h(adj_q(f, 0, k), u));
    return r;
}
// U' = M(E') U in reverse (u_adj) with Hermitian E': M^+ Yb, and e + TL of what
// E' receives
IPG_HD M3 adj_link_update(const M3& U, const H3& E, double kappa, const M3& Yb, const H3& e, H3& z) {
    const M3 Mb = mul_bd(Yb, U);
    // -i kappa Xb, Hermitian part: (-i kappa/2)(Mb - Mb^+) - (kappa^2/4) {Mb + Mb^+, E}
    z = h_traceless((e + herm_mi(0.5 * kappa, ah_of(Mb))) - (0.25 * kappa * kappa) * anticommutator(two_herm(Mb), E));
    return mul_ad(taylor2(kappa, E), Yb);
}

// ---- T^tautau at one site (lattice units, before the a^-4) ----------------------------
// e1, e1py = E1(s), E1(s+y); e2, e2px = E2(s), E2(s+x); pi at s, s+x, s+y,
// s+x+y; links for the plaquette and the phi gradients; phi at s, s+x, s+y,
// s+x+y; plaq = 0 on the last row (the reference sets U_plaq = 1 there)
struct TIn {
    M3 e1, e1py, e2, e2px, p, ppx, ppy, ppxy, ux, uy, uy_px, ux_py, ph, phpx, phpy, phpxy;
    int plaq;
};
struct TBar {
    M3 e1, e1py, e2, e2px, p, ppx, ppy, ppxy, ux, uy, uy_px, ux_py, ph, phpx, phpy, phpxy;
};
IPG_HD double tt_fwd(const TIn& q, double tau, double g) {
    const double gt = g * g / tau / tau;
    const double el = retrprod(q.e1, q.e1) + retrprod(q.e1py, q.e1py) + retrprod(q.e2, q.e2) +
                      retrprod(q.e2px, q.e2px);
    const double lng = (retrprod(q.p, q.p) + retrprod(q.ppx, q.ppx) + retrprod(q.ppy, q.ppy) +
                        retrprod(q.ppxy, q.ppxy)) /
                       4.;
    double rp = 3.;
    if (q.plaq) {
        const M3 P = (q.ux * q.uy_px) * mul_bd(dag(q.ux_py), q.uy);
        rp = tr(P).r;
    }
    const M3 dA = q.ph - q.ux * mul_bd(q.phpx, q.ux);
    const M3 dB = q.phpy - q.ux_py * mul_bd(q.phpxy, q.ux_py);
    const M3 dC = q.ph - q.uy * mul_bd(q.phpy, q.uy);
    const M3 dD = q.phpx - q.uy_px * mul_bd(q.phpxy, q.uy_px);
    const double h = 0.5 / tau / tau;
    return gt * el / 2. + lng + 2. / (g * g) * (3. - rp) +
           h * (retrprod(dA, dA) + retrprod(dB, dB) + retrprod(dC, dC) + retrprod(dD, dD));
}
IPG_HD void tt_adj(const TIn& q, double tau, double g, double yb, TBar& b) {
    const double gt = g * g / tau / tau;
    b.e1 = b.e1 + (yb * gt) * dag(q.e1);
    b.e1py = b.e1py + (yb * gt) * dag(q.e1py);
    b.e2 = b.e2 + (yb * gt) * dag(q.e2);
    b.e2px = b.e2px + (yb * gt) * dag(q.e2px);
    b.p = b.p + (yb * 0.5) * dag(q.p);
    b.ppx = b.ppx + (yb * 0.5) * dag(q.ppx);
    b.ppy = b.ppy + (yb * 0.5) * dag(q.ppy);
    b.ppxy = b.ppxy + (yb * 0.5) * dag(q.ppxy);
    if (q.plaq) {
        // d/dP of -2/g^2 Re tr P: Pb = -2/g^2 yb 1
        const M3 Pb = (-2. / (g * g) * yb) * m_one();
        M3 B1, B2, B3, B4;
        adj_prod4(q.ux, q.uy_px, dag(q.ux_py), dag(q.uy), Pb, B1, B2, B3, B4);
        b.ux = b.ux + B1;
        b.uy_px = b.uy_px + B2;
        b.ux_py = b.ux_py + dag(B3);
        b.uy = b.uy + dag(B4);
    }
    const double h2 = yb * 2. * (0.5 / tau / tau);  // d Re tr(d d) = 2 Re tr(d^+^+ dd)
    {
        const M3 d = q.ph - q.ux * mul_bd(q.phpx, q.ux);
        const M3 db = h2 * dag(d);
        b.ph = b.ph + db;
        M3 nb = -1. * db;
        adj_conj(q.ux, q.phpx, nb, b.ux, b.phpx);
    }
    {
        const M3 d = q.phpy - q.ux_py * mul_bd(q.phpxy, q.ux_py);
        const M3 db = h2 * dag(d);
        b.phpy = b.phpy + db;
        M3 nb = -1. * db;
        adj_conj(q.ux_py, q.phpxy, nb, b.ux_py, b.phpxy);
    }
    {
        const M3 d = q.ph - q.uy * mul_bd(q.phpy, q.uy);
        const M3 db = h2 * dag(d);
        b.ph = b.ph + db;
        M3 nb = -1. * db;
        adj_conj(q.uy, q.phpy, nb, b.uy, b.phpy);
    }
    {
        const M3 d = q.phpx - q.uy_px * mul_bd(q.phpxy, q.uy_px);
        const M3 db = h2 * dag(d);
        b.phpx = b.phpx + db;
        M3 nb = -1. * db;
        adj_conj(q.uy_px, q.phpxy, nb, b.uy_px, b.phpxy);
    }
}

// ---- tau = 0 root finder by implicit differentiation (Init.cpp:3344-3481) ----
// The solution U of F(U; W) = 0, F_a = -Im tr t^a [(W - W^+) + (W U^+ - U W^+)],
// lies on the coset SU(3) U0 (U = exp(i alpha t) U0, U0 = U1 U2, W = U1 + U2).
// Near it, U(beta) = exp(i beta t) E* U0 with E* = U U0^{-1}; then
//   dF_a/dbeta_b = Re tr(t^a W U^+ t^b) + Re tr(t^a t^b U W^+),
//   dU = i (dbeta . t) U + E* dU0,
// and the reverse pass is  betab_b = Re tr(Ub^+ i t^b U),
// lambda = -J^{-T} betab,  T = sum_a lambda_a t^a,
//   Wb = -2i T (1 + U) ... (from F_lambda = Re tr(i T M)),  Usb = 2i T W,
//   U0b = E*^+ (Ub + Usb),  U1b = Wb + U0b U2^+,  U2b = Wb + U1^+ U0b.
// E* = U U0^+ (U0 is unitary: products of Wilson lines).
IPG_HD void tgen(int a, M3& t) {
    t = m_zero();
    const double s3 = 1.0 / (2.0 * sqrt(3.0));
    switch (a) {
        case 0: t.e[1] = cd{0.5, 0.}; t.e[3] = cd{0.5, 0.}; break;
        case 1: t.e[1] = cd{0., -0.5}; t.e[3] = cd{0., 0.5}; break;
        case 2: t.e[0] = cd{0.5, 0.}; t.e[4] = cd{-0.5, 0.}; break;
        case 3: t.e[2] = cd{0.5, 0.}; t.e[6] = cd{0.5, 0.}; break;
        case 4: t.e[2] = cd{0., -0.5}; t.e[6] = cd{0., 0.5}; break;
        case 5: t.e[5] = cd{0.5, 0.}; t.e[7] = cd{0.5, 0.}; break;
        case 6: t.e[5] = cd{0., -0.5}; t.e[7] = cd{0., 0.5}; break;
        default: t.e[0] = cd{s3, 0.}; t.e[4] = cd{s3, 0.}; t.e[8] = cd{-2. * s3, 0.}; break;
    }
}
// solve A x = b (8x8, partial pivoting), A row-major, overwritten.  The
// loops are unrolled and the pivot rows exchanged by selects, so that A and
// b stay in registers (an exchange through a run-time row index puts them
// in scratch memory on the GPU)
IPG_HD void solve8(double (&A)[64], double (&b)[8]) {
#pragma unroll
    for (int j = 0; j < 8; j++) {
        int p = j;
        double mx = fabs(A[8 * j + j]);
#pragma unroll
        for (int r = j + 1; r < 8; r++)
            if (fabs(A[8 * r + j]) > mx) {
                mx = fabs(A[8 * r + j]);
                p = r;
            }
#pragma unroll
        for (int r = j + 1; r < 8; r++) {
            const bool sw = r == p;
#pragma unroll
            for (int c = 0; c < 8; c++) {
                const double x = A[8 * j + c], y = A[8 * r + c];
                A[8 * j + c] = sw ? y : x;
                A[8 * r + c] = sw ? x : y;
            }
            const double x = b[j], y = b[r];
            b[j] = sw ? y : x;
            b[r] = sw ? x : y;
        }
#pragma unroll
        for (int r = j + 1; r < 8; r++) {
            const double f = A[8 * r + j] / A[8 * j + j];
#pragma unroll
            for (int c = j; c < 8; c++) A[8 * r + c] -= f * A[8 * j + c];
            b[r] -= f * b[j];
        }
    }
#pragma unroll
    for (int r = 7; r >= 0; r--) {
        double t = b[r];
#pragma unroll
        for (int c = r + 1; c < 8; c++) t -= A[8 * r + c] * b[c];
        b[r] = t / A[8 * r + r];
    }
}
IPG_HD void newton_adj(const M3& U1, const M3& U2, const M3& U, const M3& Ub, M3& U1b, M3& U2b) {
    const M3 W = U1 + U2, U0 = U1 * U2;
    const M3 A = mul_bd(W, U), B = mul_bd(U, W);  // W U^+, U W^+
    // unrolled: the generators are constants, their zeros fold away
    M3 t[8];
#pragma unroll
    for (int a = 0; a < 8; a++) tgen(a, t[a]);
    double JT[64], rhs[8];  // J^T: JT[8 b + a] = J_ab
#pragma unroll
    for (int a = 0; a < 8; a++) {
        const M3 ta_A = t[a] * A;
#pragma unroll
        for (int b = 0; b < 8; b++) JT[8 * b + a] = retrprod(ta_A, t[b]) + retrprod(t[a] * t[b], B);
    }
    // betab_b = Re tr(Ub^+ i t^b U); solve J^T lambda = -betab
#pragma unroll
    for (int b = 0; b < 8; b++) {
        const M3 d = mul_i(1., t[b] * U);
        rhs[b] = -retrprod(dag(Ub), d);
    }
    solve8(JT, rhs);
    M3 T = m_zero();
#pragma unroll
    for (int a = 0; a < 8; a++) T = T + rhs[a] * t[a];
    const M3 iT = mul_i(1., T);
    const M3 Wb = (-2.) * (iT * (m_one() + U));
    const M3 Usb = 2. * (iT * W);
    const M3 Es = mul_bd(U, U0);  // E* = U U0^+
    const M3 U0b = mul_ad(Es, Ub + Usb);
    U1b = U1b + Wb + mul_bd(U0b, U2);
    U2b = U2b + Wb + mul_ad(U1, U0b);
}

// ---- pi at tau = 0: pi = -(i / 4g) acc (Init.cpp:2521-2584, 2669-2673) --------------
// x part of acc at site s from D = L1x(s) - L2x(s), U = Ux(s) and the site s-x:
//   (D U^+ - D - U D^+ + D^+) + (-U'^+ D' + D' + D'^+ U' - D'^+)
IPG_HD M3 acc_dir(const M3& D, const M3& U, const M3& Dm, const M3& Um) {
    const M3 Dd = dag(D), Dmd = dag(Dm);
    M3 acc = ((mul_bd(D, U) - D) - U * Dd) + Dd;
    return (((acc - mul_ad(Um, Dm)) + Dm) + Dmd * Um) - Dmd;
}
IPG_HD void acc_dir_adj(const M3& D, const M3& U, const M3& Dm, const M3& Um, const M3& ab, M3& Db, M3& Ub,
                        M3& Dmb, M3& Umb) {
    const M3 abd = dag(ab);
    Db = Db + ab * U - ab - abd * U + abd;
    Ub = Ub + abd * D - ab * D;
    Dmb = Dmb - Um * ab + ab + Um * abd - abd;
    Umb = Umb - Dm * abd + Dm * ab;
}

// ---- E = exp(i Q^a t^a) (Matrix.cpp:310-426): Qb_a = Re tr(Eb^+ dE/dQ_a) -------------
// By Cayley-Hamilton, exp(iQ) = f0 + f1 Q + f2 Q^2 for traceless Hermitian Q,
// the f_j being functions of c0 = det Q and c1 = tr(Q^2)/2 only
// (Morningstar and Peardon, Phys. Rev. D 69 (2004) 054501: eigenvalues 2u,
// -u+w, -u-w).  Then
//   Qb_a = Re tr(G t^a),  G = Re(b0) Q^2 + Re(b1) Q + f1 Eb^+ + f2 (Q Eb^+ + Eb^+ Q),
//   b_i = sum_j (d f_j / d c_i) tr(Eb^+ Q^j),
// from d c0 / d Q_a = tr(Q^2 t^a) and d c1 / d Q_a = tr(Q t^a).

// xi0(w) = sin(w)/w and xi1(w) = (cos w - xi0)/w^2 (Taylor series near 0)
IPG_HD void expq_xi(double w, double& x0, double& x1) {
    const double w2 = w * w;
    if (fabs(w) < 0.05) {
        x0 = 1. - w2 / 6. * (1. - w2 / 20. * (1. - w2 / 42.));
        x1 = -1. / 3. + w2 * (1. / 30. - w2 * (1. / 840. - w2 / 45360.));
    } else {
        double sw, cw;
        sincos(w, &sw, &cw);
        x0 = sw / w;
        x1 = (cw - x0) / w2;
    }
}

// f_j(c0, c1) and their partial derivatives fa_j = d/dc0, fb_j = d/dc1.
// Small c1 (all |eigenvalues| <= sqrt(4 c1 / 3) < 0.82): the exponential
// series reduced with Q^3 = c1 Q + c0; otherwise the closed form at |c0|,
// with f_j(-c0, c1) = (-1)^j conj(f_j(c0, c1)) for negative c0, which keeps
// 9u^2 - w^2 >= 2 c1 away from zero.
IPG_HD void expq_fcoef(double c0, double c1, cd (&f)[3], cd (&fa)[3], cd (&fb)[3]) {
    if (c1 < 0.5) {
        // Q^n = a I + b Q + d Q^2; (a, b, d) <- (c0 d, a + c1 d, b)
        double a = 1., b = 0., d = 0.;
        double a0 = 0., b0 = 0., d0 = 0., a1 = 0., b1 = 0., d1 = 0.;  // d/dc0, d/dc1
        double fr[3] = {0., 0., 0.}, fi[3] = {0., 0., 0.};
        double ar[3] = {0., 0., 0.}, ai[3] = {0., 0., 0.}, br[3] = {0., 0., 0.}, bi[3] = {0., 0., 0.};
        double coef = 1.;  // 1/n!
        for (int n = 0; n < 26; n++) {
            // i^n / n! = coef * (1, i, -1, -i)[n mod 4]
            const int m = n & 3;
            const double cr = m == 0 ? coef : (m == 2 ? -coef : 0.);
            const double ci = m == 1 ? coef : (m == 3 ? -coef : 0.);
            const double v[3] = {a, b, d}, v0[3] = {a0, b0, d0}, v1[3] = {a1, b1, d1};
#pragma unroll
            for (int j = 0; j < 3; j++) {
                fr[j] += cr * v[j];
                fi[j] += ci * v[j];
                ar[j] += cr * v0[j];
                ai[j] += ci * v0[j];
                br[j] += cr * v1[j];
                bi[j] += ci * v1[j];
            }
            // the recursion's matrix has 1-norm max(1, |c0| + c1) = 1 here
            // (c1 < 0.5), and its derivatives add |d| to a0 and b1, so the
            // sum s of |v|, |v0|, |v1| at most triples per term while 1/n!
            // falls at least 5-fold from n = 4: once coef s < 1e-19 the terms
            // left add less than 1.5e-19 (|f_j| is of order 1)
            const double sz = fabs(a) + fabs(b) + fabs(d) + fabs(a0) + fabs(b0) + fabs(d0) + fabs(a1) + fabs(b1) +
                              fabs(d1);
            if (n >= 4 && coef * sz < 1e-19) break;
            const double na = c0 * d, nb = a + c1 * d, nd = b;
            const double na0 = d + c0 * d0, nb0 = a0 + c1 * d0, nd0 = b0;
            const double na1 = c0 * d1, nb1 = a1 + d + c1 * d1, nd1 = b1;
            a = na, b = nb, d = nd;
            a0 = na0, b0 = nb0, d0 = nd0;
            a1 = na1, b1 = nb1, d1 = nd1;
            coef /= (double)(n + 1);
        }
#pragma unroll
        for (int j = 0; j < 3; j++) {
            f[j] = cd{fr[j], fi[j]};
            fa[j] = cd{ar[j], ai[j]};
            fb[j] = cd{br[j], bi[j]};
        }
        return;
    }
    const bool neg = c0 < 0.;
    const double c0p = fabs(c0);
    const double x3 = c1 / 3.;
    const double c0max = 2. * x3 * sqrt(x3);
    const double th = acos(fmin(c0p / c0max, 1.)) / 3.;
    double sth, cth;
    sincos(th, &sth, &cth);
    const double u = sqrt(x3) * cth, w = sqrt(c1) * sth;
    double x0, x1;
    expq_xi(w, x0, x1);
    const double cw = cos(w), u2 = u * u, w2 = w * w;
    double s2u, c2u, su, cu;
    sincos(2. * u, &s2u, &c2u);
    sincos(u, &su, &cu);
    const cd e2{c2u, s2u}, em{cu, -su};
    // h_j = D f_j, D = 9u^2 - w^2; hu = dh/du; hw = (1/w) dh/dw
    cd h[3], hu[3], hw[3];
    h[0] = e2 * (u2 - w2) + em * cd{8. * u2 * cw, 2. * u * (3. * u2 + w2) * x0};
    h[1] = e2 * (2. * u) - em * cd{2. * u * cw, -(3. * u2 - w2) * x0};
    h[2] = e2 - em * cd{cw, 3. * u * x0};
    hu[0] = e2 * cd{2. * u, 2. * (u2 - w2)} +
            em * cd{16. * u * cw + 2. * u * (3. * u2 + w2) * x0, -8. * u2 * cw + 2. * (9. * u2 + w2) * x0};
    hw[0] = e2 * (-2.) + em * cd{-8. * u2 * x0, 2. * u * (2. * x0 + (3. * u2 + w2) * x1)};
    hu[1] = e2 * cd{2., 4. * u} + em * cd{(3. * u2 - w2) * x0 - 2. * cw, 2. * u * cw + 6. * u * x0};
    hw[1] = em * cd{2. * u * x0, -2. * x0 + (3. * u2 - w2) * x1};
    hu[2] = e2 * cd{0., 2.} + em * cd{-3. * u * x0, cw - 3. * x0};
    hw[2] = em * cd{x0, -3. * u * x1};
    const double D = 9. * u2 - w2;
    const double iD = 1. / D;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        f[j] = h[j] * iD;
        const cd fu = (hu[j] - f[j] * (18. * u)) * iD;
        const cd fw = (hw[j] + f[j] * 2.) * iD;
        fa[j] = (fu - fw * (3. * u)) * (0.5 * iD);
        fb[j] = fu * (u * iD) + fw * ((3. * u2 - w2) * 0.5 * iD);
    }
    if (neg) {
        // f_j(-c0) = (-1)^j conj f_j(c0); d/dc0 picks up one more sign
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const double sj = (j & 1) ? -1. : 1.;
            f[j] = cd{sj * f[j].r, -sj * f[j].i};
            fa[j] = cd{-sj * fa[j].r, sj * fa[j].i};
            fb[j] = cd{sj * fb[j].r, -sj * fb[j].i};
        }
    }
}

// Q = Q^a t^a, t^a = lambda^a / 2 (Gell-Mann order)
IPG_HD M3 gen_matrix(const double (&Q)[8]) {
    const double s3 = 1. / (2. * sqrt(3.));
    M3 m;
    m.e[0] = cd{0.5 * Q[2] + s3 * Q[7], 0.};
    m.e[4] = cd{-0.5 * Q[2] + s3 * Q[7], 0.};
    m.e[8] = cd{-2. * s3 * Q[7], 0.};
    m.e[1] = cd{0.5 * Q[0], -0.5 * Q[1]};
    m.e[3] = cd{0.5 * Q[0], 0.5 * Q[1]};
    m.e[2] = cd{0.5 * Q[3], -0.5 * Q[4]};
    m.e[6] = cd{0.5 * Q[3], 0.5 * Q[4]};
    m.e[5] = cd{0.5 * Q[5], -0.5 * Q[6]};
    m.e[7] = cd{0.5 * Q[5], 0.5 * Q[6]};
    return m;
}
// Re tr(G t^a), a = 0..7
IPG_HD void gen_project(const M3& G, double (&out)[8]) {
    const double s3 = 1. / (2. * sqrt(3.));
    out[0] = 0.5 * (G.e[1].r + G.e[3].r);
    out[1] = 0.5 * (G.e[3].i - G.e[1].i);
    out[2] = 0.5 * (G.e[0].r - G.e[4].r);
    out[3] = 0.5 * (G.e[2].r + G.e[6].r);
    out[4] = 0.5 * (G.e[6].i - G.e[2].i);
    out[5] = 0.5 * (G.e[5].r + G.e[7].r);
    out[6] = 0.5 * (G.e[7].i - G.e[5].i);
    out[7] = s3 * (G.e[0].r + G.e[4].r - 2. * G.e[8].r);
}

// exp(i Q^a t^a) = f0 + f1 Q + f2 Q^2 and what its reverse needs: Q, Q^2,
// the coefficients f_j(c0, c1) and their derivatives (computed once when a
// caller wants both the exponential and its reverse)
struct ExpQ {
    M3 Qm, Q2;
    cd f[3], fa[3], fb[3];
};
IPG_HD void expq_prep(const double (&Q)[8], ExpQ& x) {
    x.Qm = gen_matrix(Q);
    x.Q2 = x.Qm * x.Qm;
    double c1 = 0.;
#pragma unroll
    for (int a = 0; a < 8; a++) c1 += Q[a] * Q[a];
    c1 *= 0.25;
    const double c0 = retrprod(x.Q2, x.Qm) / 3.;  // det Q = tr(Q^3) / 3
    expq_fcoef(c0, c1, x.f, x.fa, x.fb);
}
// the exponential from the coefficients (equal to exp_iQt to round-off)
IPG_HD M3 expq_value(const ExpQ& x) {
    M3 E = cscale(x.f[1], x.Qm) + cscale(x.f[2], x.Q2);
    E.e[0] = E.e[0] + x.f[0];
    E.e[4] = E.e[4] + x.f[0];
    E.e[8] = E.e[8] + x.f[0];
    return E;
}
// The setV slices' exponential exp(i Q^a t^a) without its reverse: the
// Cayley-Hamilton form f0 + f1 Q + f2 Q^2 with the f_j summed as the series
// of exp(i x) in the basis {1, Q, Q^2} (Q^3 = c0 + c1 Q) for c1 = tr(Q^2)/2
// below kExpqSeriesMax, stopped once the terms left are below 1.5e-19 (the
// bound of expq_fcoef); larger Q scaled into that range and the factor
// applied repeatedly (expq_apply).  No transcendental functions.  It agrees
// with exp_iQt's closed form (Matrix.cpp:310-426) to round-off except at
// (nearly) degenerate spectra, where the closed form loses digits or
// returns 1, and at |Q| below ~1e-8, where the closed form cancels
// catastrophically (its 9u^2 - w^2 denominator and a floor of 1e-15 on
// c0max) and its value, off the exponential by up to |Q|, depends on the
// last bits of acos and sincos.
constexpr double kExpqSeriesMax = 0.5;
// the f_j of the series: exp(i x) summed in the basis {1, Q, Q^2} with
// Q^3 = c0 + c1 Q (the powers Q^n = a_n + b_n Q + d_n Q^2)
IPG_HD void expq_series(double c0, double c1, cd (&f)[3]) {
    double a = 1., b = 0., d = 0.;
    double fr[3] = {0., 0., 0.}, fi[3] = {0., 0., 0.};
    double coef = 1.;  // 1/n!
    for (int n = 0; n < 26; n++) {
        const int m = n & 3;
        const double cr = m == 0 ? coef : (m == 2 ? -coef : 0.);
        const double ci = m == 1 ? coef : (m == 3 ? -coef : 0.);
        fr[0] += cr * a;
        fi[0] += ci * a;
        fr[1] += cr * b;
        fi[1] += ci * b;
        fr[2] += cr * d;
        fi[2] += ci * d;
        if (n >= 4 && coef * (fabs(a) + fabs(b) + fabs(d)) < 1e-19) break;
        const double na = c0 * d, nb = a + c1 * d, nd = b;
        a = na, b = nb, d = nd;
        coef /= (double)(n + 1);
    }
#pragma unroll
    for (int j = 0; j < 3; j++) f[j] = cd{fr[j], fi[j]};
}
// det(Q^a t^a) from the components (gen_matrix's entries: real diagonal
// d_i, upper triangle q01, q02, q12):
// d0 d1 d2 - d0 |q12|^2 - d1 |q02|^2 - d2 |q01|^2 + 2 Re(q01 q12 conj q02)
IPG_HD double gen_det(const double (&Q)[8]) {
    const double s3 = 1. / (2. * sqrt(3.));
    const double d0 = 0.5 * Q[2] + s3 * Q[7], d1 = -0.5 * Q[2] + s3 * Q[7], d2 = -2. * s3 * Q[7];
    const cd q01{0.5 * Q[0], -0.5 * Q[1]}, q02{0.5 * Q[3], -0.5 * Q[4]}, q12{0.5 * Q[5], -0.5 * Q[6]};
    const double n01 = q01.r * q01.r + q01.i * q01.i, n02 = q02.r * q02.r + q02.i * q02.i,
                 n12 = q12.r * q12.r + q12.i * q12.i;
    return d0 * d1 * d2 - d0 * n12 - d1 * n02 - d2 * n01 + 2. * mulc(q01 * q12, q02).r;
}
// V <- (f0 + f1 Q + f2 Q^2) V column by column: v <- f0 v + f1 (Q v) +
// f2 Q (Q v), Q = Q^a t^a from its components.  Neither Q^2 nor the
// exponential is formed, so far fewer values are live than in E * V.
IPG_HD void expq_coef_apply(const double (&Q)[8], const cd (&f)[3], M3& V) {
    const double s3 = 1. / (2. * sqrt(3.));
    const double d0 = 0.5 * Q[2] + s3 * Q[7], d1 = -0.5 * Q[2] + s3 * Q[7], d2 = -2. * s3 * Q[7];
    const cd q01{0.5 * Q[0], -0.5 * Q[1]}, q02{0.5 * Q[3], -0.5 * Q[4]}, q12{0.5 * Q[5], -0.5 * Q[6]};
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const cd v0 = V.e[j], v1 = V.e[3 + j], v2 = V.e[6 + j];
        const cd w0 = v0 * d0 + q01 * v1 + q02 * v2;
        const cd w1 = cmul(q01, v0) + v1 * d1 + q12 * v2;
        const cd w2 = cmul(q02, v0) + cmul(q12, v1) + v2 * d2;
        const cd x0 = w0 * d0 + q01 * w1 + q02 * w2;
        const cd x1 = cmul(q01, w0) + w1 * d1 + q12 * w2;
        const cd x2 = cmul(q02, w0) + cmul(q12, w1) + w2 * d2;
        V.e[j] = f[0] * v0 + f[1] * w0 + f[2] * x0;
        V.e[3 + j] = f[0] * v1 + f[1] * w1 + f[2] * x1;
        V.e[6 + j] = f[0] * v2 + f[1] * w2 + f[2] * x2;
    }
}
// V <- exp(i Q^a t^a) V for any Q (the setV slices): Q scaled by 2^-s
// (exact) until c1 = tr(Q^2)/2 is below kExpqSeriesMax, the series
// coefficients of the scaled Q (expq_series, c0 = det Q), applied 2^s times
// by expq_coef_apply.  No transcendental functions; s is at most 12
// (c1 < 8.4e6), so that no input can make the loop long.
IPG_HD void expq_apply(const double (&Q)[8], M3& V) {
    double c1 = 0.;
#pragma unroll
    for (int a = 0; a < 8; a++) c1 += Q[a] * Q[a];
    c1 *= 0.25;
    double sc = 1.;
    int reps = 1;
    while (c1 >= kExpqSeriesMax && reps < 4096) {
        c1 *= 0.25;
        sc *= 0.5;
        reps *= 2;
    }
    double Qs[8];
#pragma unroll
    for (int a = 0; a < 8; a++) Qs[a] = Q[a] * sc;
    cd f[3];
    expq_series(gen_det(Qs), c1, f);
    for (int r = 0; r < reps; r++) expq_coef_apply(Qs, f, V);
}
// the slice exponential itself (expq_apply to the identity)
IPG_HD M3 expq_forward(const double (&Q)[8]) {
    M3 E = m_one();
    expq_apply(Q, E);
    return E;
}
// Qb^a = Re tr(Eb^+ dE/dQ^a)
IPG_HD void expq_back(const ExpQ& x, const M3& Eb, double (&Qb)[8]) {
    const M3 Ebd = dag(Eb);
    const cd t0 = tr(Ebd), t1 = trprod(Ebd, x.Qm), t2 = trprod(Ebd, x.Q2);
    const double b0 = (x.fa[0] * t0 + x.fa[1] * t1 + x.fa[2] * t2).r;
    const double b1 = (x.fb[0] * t0 + x.fb[1] * t1 + x.fb[2] * t2).r;
    const M3 G = (b0 * x.Q2 + b1 * x.Qm) + (cscale(x.f[1], Ebd) + cscale(x.f[2], x.Qm * Ebd + Ebd * x.Qm));
    gen_project(G, Qb);
}
IPG_HD void expq_adj(const double (&Q)[8], const M3& Eb, double (&Qb)[8]) {
    ExpQ x;
    expq_prep(Q, x);
    expq_back(x, Eb, Qb);
}

}  // namespace ipgad


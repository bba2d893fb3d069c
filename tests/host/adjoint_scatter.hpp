// The pi and E updates of one leapfrog step at one site, forward, and in reverse
// as cotangents scattered to the sites of the stencil: what the kernels' gathered
// sums (ipglasma_amd/csrc/adjoint.hpp) are checked against.
#pragma once
#include "../../ipglasma_amd/csrc/adjoint.hpp"

namespace ipgad {

// ---- pi update -------------------------------------------------------------------
// inputs of site s: ux = Ux(s), uy = Uy(s), uxm = Ux(s-x), uym = Uy(s-y),
// phi at s, s+x, s-x, s+y, s-y; cp = dtau/tau
struct PiIn {
    M3 ux, uy, uxm, uym, ph, phpx, phmx, phpy, phmy, pi;
};
IPG_HD M3 pi_fwd(const PiIn& q, double cp) {
    const M3 br = (((q.ux * mul_bd(q.phpx, q.ux) + mul_ad(q.uxm, q.phmx) * q.uxm) + q.uy * mul_bd(q.phpy, q.uy)) +
                   mul_ad(q.uym, q.phmy) * q.uym) -
                  4. * q.ph;
    return q.pi + cp * br;
}
struct PiBar {
    M3 ux, uy, uxm, uym, ph, phpx, phmx, phpy, phmy, pi;
};
IPG_HD void pi_adj(const PiIn& q, double cp, const M3& Yb, PiBar& b) {
    b.pi = b.pi + Yb;
    const M3 Bb = cp * Yb;
    adj_conj(q.ux, q.phpx, Bb, b.ux, b.phpx);
    adj_conjd(q.uxm, q.phmx, Bb, b.uxm, b.phmx);
    adj_conj(q.uy, q.phpy, Bb, b.uy, b.phpy);
    adj_conjd(q.uym, q.phmy, Bb, b.uym, b.phmy);
    b.ph = b.ph - 4. * Bb;
}

// ---- E update -----------------------------------------------------------------------
// links: ux, uy at s; uy_px = Uy(s+x), ux_py = Ux(s+y), uy_pxmy = Uy(s+x-y),
// ux_my = Ux(s-y), uy_my = Uy(s-y), ux_mxpy = Ux(s-x+y), uy_mx = Uy(s-x),
// ux_mx = Ux(s-x); phi at s, s+x, s+y
struct EIn {
    M3 ux, uy, uy_px, ux_py, uy_pxmy, ux_my, uy_my, ux_mxpy, uy_mx, ux_mx, ph, phpx, phpy, e1, e2;
};
struct EBar {
    M3 ux, uy, uy_px, ux_py, uy_pxmy, ux_my, uy_my, ux_mxpy, uy_mx, ux_mx, ph, phpx, phpy, e1, e2;
};
IPG_HD void e_fwd(const EIn& q, double tau, double dtau, double g, M3& e1n, M3& e2n) {
    const cd c1{0., tau * dtau / (2. * g * g)}, c2{0., dtau / tau};
    const M3 U12 = (q.ux * q.uy_px) * mul_bd(dag(q.ux_py), q.uy);
    const M3 U1m2 = mul_bd(q.ux, q.uy_pxmy) * mul_ad(q.ux_my, q.uy_my);
    const M3 U2m1 = mul_bd(q.uy, q.ux_mxpy) * mul_ad(q.uy_mx, q.ux_mx);
    const M3 tx = q.ux * mul_bd(q.phpx, q.ux), ty = q.uy * mul_bd(q.phpy, q.uy);
    M3 t1 = traceless(((U12 + U1m2) - dag(U12)) - dag(U1m2));
    M3 t2 = tx * q.ph - q.ph * tx;
    e1n = traceless(q.e1 + (cscale(c1, t1) + cscale(c2, t2)));
    t1 = traceless(((dag(U12) + U2m1) - U12) - dag(U2m1));
    t2 = ty * q.ph - q.ph * ty;
    e2n = traceless(q.e2 + (cscale(c1, t1) + cscale(c2, t2)));
}
// the E' update in reverse, in pieces: Z1, Z2 = TL(E1'b), TL(E2'b) give the
// cotangents of the three plaquette products U12, U1m2, U2m1 ...
IPG_HD void plaq_bars(const M3& Z1, const M3& Z2, double tau, double dtau, double g, M3& U12b, M3& U1m2b,
                      M3& U2m1b) {
    const cd c1c{0., -tau * dtau / (2. * g * g)};  // conj(c1)
    const M3 t1b = traceless(cscale(c1c, Z1)), t1pb = traceless(cscale(c1c, Z2));
    // t1 = U12 + U1m2 - U12^+ - U1m2^+, t1' = U12^+ + U2m1 - U12 - U2m1^+
    U12b = (t1b - dag(t1b)) + (dag(t1pb) - t1pb);
    U1m2b = t1b - dag(t1b);
    U2m1b = t1pb - dag(t1pb);
}
// ... and, with t2b = conj(c2) Z, the commutator t2 = tx phi - phi tx,
// tx = U phn U^+ (tx, phi Hermitian): cotangents of phi, U and phn
IPG_HD void comm_adj(const M3& U, const M3& phn, const M3& ph, const M3& t2b, M3& phb, M3& Ub, M3& phnb) {
    const M3 tx = U * mul_bd(phn, U);
    const M3 txb = t2b * ph - ph * t2b;
    phb = phb + (tx * t2b - t2b * tx);
    adj_conj(U, phn, txb, Ub, phnb);
}
IPG_HD void e_adj(const EIn& q, double tau, double dtau, double g, const M3& Y1b, const M3& Y2b, EBar& b) {
    const cd c2c{0., -dtau / tau};  // conj(c2)
    const M3 Z1 = traceless(Y1b), Z2 = traceless(Y2b);
    b.e1 = b.e1 + Z1;
    b.e2 = b.e2 + Z2;
    M3 U12b, U1m2b, U2m1b;
    plaq_bars(Z1, Z2, tau, dtau, g, U12b, U1m2b, U2m1b);
    M3 B1, B2, B3, B4;
    // U12 = ux uy_px ux_py^+ uy^+
    adj_prod4(q.ux, q.uy_px, dag(q.ux_py), dag(q.uy), U12b, B1, B2, B3, B4);
    b.ux = b.ux + B1;
    b.uy_px = b.uy_px + B2;
    b.ux_py = b.ux_py + dag(B3);
    b.uy = b.uy + dag(B4);
    // U1m2 = ux uy_pxmy^+ ux_my^+ uy_my
    adj_prod4(q.ux, dag(q.uy_pxmy), dag(q.ux_my), q.uy_my, U1m2b, B1, B2, B3, B4);
    b.ux = b.ux + B1;
    b.uy_pxmy = b.uy_pxmy + dag(B2);
    b.ux_my = b.ux_my + dag(B3);
    b.uy_my = b.uy_my + B4;
    // U2m1 = uy ux_mxpy^+ uy_mx^+ ux_mx
    adj_prod4(q.uy, dag(q.ux_mxpy), dag(q.uy_mx), q.ux_mx, U2m1b, B1, B2, B3, B4);
    b.uy = b.uy + B1;
    b.ux_mxpy = b.ux_mxpy + dag(B2);
    b.uy_mx = b.uy_mx + dag(B3);
    b.ux_mx = b.ux_mx + B4;
    comm_adj(q.ux, q.phpx, q.ph, cscale(c2c, Z1), b.ph, b.ux, b.phpx);
    comm_adj(q.uy, q.phpy, q.ph, cscale(c2c, Z2), b.ph, b.uy, b.phpy);
}

}  // namespace ipgad

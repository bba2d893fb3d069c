// Host build of the reverse step of ipglasma_amd/csrc/adjoint.hpp on a small
// clamped lattice: the cotangents gathered per site (what the kernels run)
// beside the same sums scattered site by site with e_adj and pi_adj.
#include <algorithm>
#include <vector>

#include "adjoint_scatter.hpp"

using namespace ipgad;

namespace {
M3 ld(const double* p) {
    M3 m;
    for (int k = 0; k < 9; k++) m.e[k] = cd{p[2 * k], p[2 * k + 1]};
    return m;
}
void st(double* p, const M3& m) {
    for (int k = 0; k < 9; k++) {
        p[2 * k] = m.e[k].r;
        p[2 * k + 1] = m.e[k].i;
    }
}
H3 ldh(const double* p) {
    const M3 m = ld(p);
    H3 h;
    for (int k = 0; k < 3; k++) h.d[k] = m.e[4 * k].r;
    h.o[0] = m.e[1];
    h.o[1] = m.e[2];
    h.o[2] = m.e[5];
    return h;
}
M3 full(const H3& h) {
    M3 m;
    for (int k = 0; k < 3; k++) m.e[4 * k] = cd{h.d[k], 0.};
    m.e[1] = h.o[0];
    m.e[2] = h.o[1];
    m.e[5] = h.o[2];
    m.e[3] = cconj(h.o[0]);
    m.e[6] = cconj(h.o[1]);
    m.e[7] = cconj(h.o[2]);
    return m;
}
// fields [N*N][18] at the clamped offset (dp, dq) from the site (i, j); dir 0:
// (p, q) = (i, j), 1: (j, i)
struct Acc {
    int N, dir, p, q;
    double k;
    const double *ux, *uy, *z1, *z2, *phi, *pib;
    const double* at(const double* f, int dp, int dq) const {
        const int a = std::min(std::max(p + dp, 0), N - 1), b = std::min(std::max(q + dq, 0), N - 1);
        return f + 18 * (dir ? b * N + a : a * N + b);
    }
    M3 uf(int dp, int dq) const { return ld(at(dir ? uy : ux, dp, dq)); }
    M3 uo(int dp, int dq) const { return ld(at(dir ? ux : uy, dp, dq)); }
    H3 zf(int dp, int dq) const { return ldh(at(dir ? z2 : z1, dp, dq)); }
    H3 zo(int dp, int dq) const { return ldh(at(dir ? z1 : z2, dp, dq)); }
    H3 ph(int dp, int dq) const { return ldh(at(phi, dp, dq)); }
    H3 bb(int dp, int dq) const { return k * ldh(at(pib, dp, dq)); }
};
M3 link(const Acc& f, double a) {
    return mul_i(-2. * a, adj_link_above(f) + adj_link_below(f)) + adj_link_phi(f, f.k);
}
}  // namespace

// out, ref: [3][N*N][18], the cotangents of U_x, U_y and phi (Hermitian part)
extern "C" void adj_gather_host(int N, double tau, double dtau, double g, const double* ux, const double* uy,
                                const double* phi, const double* z1, const double* z2, const double* pib, double* out,
                                double* ref) {
    const size_t F = 18 * (size_t)N * N;
    const double a = tau * dtau / (2. * g * g), k = dtau / tau;
    for (int i = 0; i < N; i++)
        for (int j = 0; j < N; j++) {
            const Acc fx{N, 0, i, j, k, ux, uy, z1, z2, phi, pib};
            const Acc fy{N, 1, j, i, k, ux, uy, z1, z2, phi, pib};
            double* o = out + 18 * (i * N + j);
            st(o, link(fx, a));
            st(o + F, link(fy, a));
            st(o + 2 * F, full(((-4.) * fx.bb(0, 0) + adj_phi_dir(fx, k)) + adj_phi_dir(fy, k)));
        }
    auto cl = [&](int v) { return v < 0 ? 0 : (v > N - 1 ? N - 1 : v); };
    std::vector<M3> u1(N * N, m_zero()), u2(N * N, m_zero()), ph(N * N, m_zero());
    for (int i = 0; i < N; i++)
        for (int j = 0; j < N; j++) {
            auto at = [&](int di, int dj) { return cl(i + di) * N + cl(j + dj); };
            const int s = at(0, 0), pX = at(1, 0), pY = at(0, 1), mX = at(-1, 0), mY = at(0, -1);
            const int pXmY = at(1, -1), mXpY = at(-1, 1);
            auto L = [&](const double* f, int q) { return ld(f + 18 * q); };
            EIn e{L(ux, s),    L(uy, s),  L(uy, pX),  L(ux, pY),  L(uy, pXmY), L(ux, mY), L(uy, mY),   L(ux, mXpY),
                  L(uy, mX),   L(ux, mX), L(phi, s),  L(phi, pX), L(phi, pY),  m_zero(),  m_zero()};
            EBar b{};
            e_adj(e, tau, dtau, g, L(z1, s), L(z2, s), b);
            u1[s] = u1[s] + b.ux;
            u2[s] = u2[s] + b.uy;
            u2[pX] = u2[pX] + b.uy_px;
            u1[pY] = u1[pY] + b.ux_py;
            u2[pXmY] = u2[pXmY] + b.uy_pxmy;
            u1[mY] = u1[mY] + b.ux_my;
            u2[mY] = u2[mY] + b.uy_my;
            u1[mXpY] = u1[mXpY] + b.ux_mxpy;
            u2[mX] = u2[mX] + b.uy_mx;
            u1[mX] = u1[mX] + b.ux_mx;
            ph[s] = ph[s] + b.ph;
            ph[pX] = ph[pX] + b.phpx;
            ph[pY] = ph[pY] + b.phpy;
            PiIn q{L(ux, s),   L(uy, s),   L(ux, mX),  L(uy, mY),  L(phi, s), L(phi, pX),
                   L(phi, mX), L(phi, pY), L(phi, mY), m_zero()};
            PiBar c{};
            pi_adj(q, k, L(pib, s), c);
            u1[s] = u1[s] + c.ux;
            u2[s] = u2[s] + c.uy;
            u1[mX] = u1[mX] + c.uxm;
            u2[mY] = u2[mY] + c.uym;
            ph[s] = ph[s] + c.ph;
            ph[pX] = ph[pX] + c.phpx;
            ph[mX] = ph[mX] + c.phmx;
            ph[pY] = ph[pY] + c.phpy;
            ph[mY] = ph[mY] + c.phmy;
        }
    for (int s = 0; s < N * N; s++) {
        st(ref + 18 * s, u1[s]);
        st(ref + F + 18 * s, u2[s]);
        st(ref + 2 * F + 18 * s, hproj(ph[s]));
    }
}
// U' = M(E') U in reverse: adj_link_update beside u_adj with the projections
// the step applies; out, ref: [2][18] (M^+ Yb, TL of the E' cotangent)
extern "C" void adj_link_update_host(const double* u, const double* e, double kappa, const double* yb, const double* eb,
                                     double* out, double* ref) {
    H3 z;
    st(out, adj_link_update(ld(u), ldh(e), kappa, ld(yb), ldh(eb), z));
    st(out + 18, full(z));
    M3 Ub = m_zero(), Eb = ld(eb);
    u_adj(ld(u), ld(e), kappa, ld(yb), Ub, Eb);
    st(ref, Ub);
    st(ref + 18, traceless(hproj(Eb)));
}

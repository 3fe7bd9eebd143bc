// helgrad_check.cpp -- TEST INFRASTRUCTURE ONLY: the adjoint's closed-form
// helicity gradients (3photons-rust_amd/csrc/tp_helicity.h, built here for the
// host) and the reference's spinor-product sums (spinor.rs:31-162,
// matelems.rs:53-86) on dual numbers over long double.
//
//   g++ -O2 -std=c++17 -ffp-contract=off -shared -fPIC -I<csrc> helgrad_check.cpp
#include <cmath>

#include "tp_helicity.h"

typedef long double L;

namespace {
struct D { // value and one directional derivative
    L v, d;
};
D operator+(D a, D b) { return {a.v + b.v, a.d + b.d}; }
D operator-(D a, D b) { return {a.v - b.v, a.d - b.d}; }
D operator*(D a, D b) { return {a.v * b.v, a.v * b.d + a.d * b.v}; }
D operator/(D a, D b) { return {a.v / b.v, (a.d - a.v / b.v * b.d) / b.v}; }
D root(D a)
{
    const L r = std::sqrt(a.v);
    return {r, a.d / (2 * r)};
}
struct Z {
    D re, im;
};
Z operator+(Z a, Z b) { return {a.re + b.re, a.im + b.im}; }
Z operator-(Z a, Z b) { return {a.re - b.re, a.im - b.im}; }
Z operator*(Z a, Z b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
Z conj(Z a) { return {a.re, D{0, 0} - a.im}; }
D norm(Z a) { return a.re * a.re + a.im * a.im; }
Z operator/(Z a, Z b)
{
    const Z n = a * conj(b);
    return {n.re / norm(b), n.im / norm(b)};
}
Z real(L x) { return {{x, 0}, {0, 0}}; }
Z sq(Z a) { return a * a; }
} // namespace

// m[n][5], g[n][5][3][4] (d/dX, Y, Z, E) of momenta p[n][3][4].
extern "C" void tp_helgrad_closed(double e, double ga, double gp, double gm, long n, const double *p, double *m, double *g)
{
    const tpd::HelicityK K = tpd::helicity_constants(e, ga, gp, gm, 1.);
    for (long i = 0; i < n; ++i) {
        const double(*q)[4] = reinterpret_cast<const double(*)[4]>(p + 12 * i);
        double gg[5][3][3];
        int along;
        tpd::helicity_gradients(K, q, m + 5 * i, gg, along);
        for (int c = 0; c < 5; ++c)
            for (int k = 0; k < 3; ++k) {
                double *o = g + 60 * i + 12 * c + 4 * k;
                o[0] = gg[c][k][0];
                o[1] = gg[c][k][1];
                o[2] = along >> k & 1 ? 0. : gg[c][k][2];
                o[3] = gg[c][k][2];
            }
    }
}

extern "C" void tp_helgrad_spinors(double e, double ga, double gp, double gm, long n, const double *P, double *M, double *G)
{
    for (long i = 0; i < n; ++i)
        for (int dir = 0; dir < 12; ++dir) {
            D p[3][4];
            for (int k = 0; k < 12; ++k)
                p[k / 4][k % 4] = D{P[12 * i + k], k == dir ? 1.L : 0.L};
            Z xx[5], f[5], s[5][5], t[5][5];
            xx[0] = xx[1] = real(std::sqrt((L)e / 2));
            f[0] = real(-std::sqrt((L)e / 2));
            f[1] = real(std::sqrt((L)e / 2));
            for (int k = 0; k < 3; ++k) {
                if (p[k][3].v + p[k][2].v > 0) {
                    const D r = root(p[k][3] + p[k][2]);
                    xx[2 + k] = Z{r, {0, 0}};
                    f[2 + k] = Z{p[k][0] / r, p[k][1] / r};
                } else { // a photon along -Z: (0, sqrt(2E)), with no derivative of sqrt(E + Z)
                    xx[2 + k] = real(0);
                    f[2 + k] = Z{root(p[k][3] + p[k][3]), {0, 0}};
                }
            }
            for (int a = 0; a < 5; ++a)
                for (int b = 0; b < 5; ++b) {
                    s[a][b] = f[a] * xx[b] - f[b] * xx[a];
                    t[a][b] = real(0) - conj(s[a][b]);
                }
            const Z ns = real(-2 * std::sqrt((L)2)) * s[0][1], nt = real(-2 * std::sqrt((L)2)) * t[0][1];
            D mA{0, 0}, mP{0, 0};
            Z X = real(0);
            const int T[3][3] = {{2, 3, 4}, {2, 4, 3}, {3, 4, 2}};
            for (const auto &q : T) {
                const int a = q[0], b = q[1], c = q[2];
                const Z A1 = real(ga) * ns * sq(s[0][c]) / (s[0][a] * s[0][b] * s[1][a] * s[1][b]);
                const Z B1 = real(gp) * nt * sq(t[a][b] * s[c][0]);
                const Z A2 = real(ga) * nt * sq(t[1][c]) / (t[1][a] * t[1][b] * t[0][a] * t[0][b]);
                const Z B2 = real(gp) * ns * sq(t[c][1] * s[a][b]);
                mA = mA + norm(A1) + norm(A2);
                mP = mP + norm(B1) + norm(B2);
                X = X + real(2) * (A1 * conj(B1) + A2 * conj(B2));
            }
            const Z Bp = real(gm) * ns * (sq(t[2][3] * t[4][1]) + sq(t[2][4] * t[3][1]) + sq(t[3][4] * t[2][1]));
            const Z Bm = real(gm) * nt * (sq(s[2][0] * s[3][4]) + sq(s[3][0] * s[2][4]) + sq(s[4][0] * s[2][3]));
            const D r[5] = {mA, mP, norm(Bp) + norm(Bm), X.re, X.im};
            for (int c = 0; c < 5; ++c) {
                M[5 * i + c] = (double)r[c].v;
                G[60 * i + 12 * c + dir] = (double)r[c].d;
            }
        }
}

// helicity_check.cpp -- TEST INFRASTRUCTURE ONLY: the event loop's closed-form
// helicity sums (3photons-rust_amd/csrc/tp_helicity.h, built here for the host)
// and the reference's spinor-product amplitudes (spinor.rs:31-162,
// matelems.rs:53-86) in long double, on given photon momenta.
//
//   g++ -O2 -std=c++17 -ffp-contract=off -shared -fPIC -I<csrc> helicity_check.cpp
#include <cmath>
#include <complex>

#include "tp_helicity.h"

typedef long double L;
typedef std::complex<L> CL;

// m[n][5] of momenta p[n][3][4] times the engine's energy unit for e.
extern "C" void tp_helicity_closed(double e, double ga, double gp, double gm, long n, const double *p, double *m)
{
    const double u = tpd::energy_unit(e);
    const tpd::HelicityK K = tpd::helicity_constants(e, ga, gp, gm, u);
    for (long i = 0; i < n; ++i) {
        double q[3][4];
        for (int k = 0; k < 12; ++k)
            q[k / 4][k % 4] = p[12 * i + k] * u;
        tpd::helicity_sums_closed(K, q, m + 5 * i);
    }
}

extern "C" void tp_helicity_spinors(double e, double ga, double gp, double gm, long n, const double *P, double *M)
{
    auto sq = [](CL z) { return z * z; };
    for (long i = 0; i < n; ++i) {
        const double(*p)[4] = reinterpret_cast<const double(*)[4]>(P + 12 * i);
        double *m = M + 5 * i;
        L xx[5];
        CL f[5], s[5][5], t[5][5];
        xx[0] = xx[1] = std::sqrt((L)e / 2);
        f[0] = -((L)e / 2) / xx[0];
        f[1] = ((L)e / 2) / xx[1];
        for (int k = 0; k < 3; ++k) {
            xx[2 + k] = std::sqrt((L)p[k][3] + (L)p[k][2]);
            f[2 + k] = xx[2 + k] > 0 ? CL(p[k][0], p[k][1]) / xx[2 + k] : CL(std::sqrt(2 * (L)p[k][3]), 0);
        }
        for (int a = 0; a < 5; ++a)
            for (int b = 0; b < 5; ++b) {
                s[a][b] = f[a] * xx[b] - f[b] * xx[a];
                t[a][b] = -std::conj(s[a][b]);
            }
        const L r8 = -2 * std::sqrt((L)2);
        const CL ns = r8 * s[0][1], nt = r8 * t[0][1];
        L mA = 0, mP = 0;
        CL X = 0;
        const int T[3][3] = {{2, 3, 4}, {2, 4, 3}, {3, 4, 2}};
        for (const auto &q : T) {
            const int a = q[0], b = q[1], c = q[2];
            const CL A1 = (L)ga * ns * sq(s[0][c]) / (s[0][a] * s[0][b] * s[1][a] * s[1][b]);
            const CL B1 = (L)gp * nt * sq(t[a][b] * s[c][0]);
            const CL A2 = (L)ga * nt * sq(t[1][c]) / (t[1][a] * t[1][b] * t[0][a] * t[0][b]);
            const CL B2 = (L)gp * ns * sq(t[c][1] * s[a][b]);
            mA += std::norm(A1) + std::norm(A2);
            mP += std::norm(B1) + std::norm(B2);
            X += (L)2 * (A1 * std::conj(B1) + A2 * std::conj(B2));
        }
        const CL Bp = (L)gm * ns * (sq(t[2][3] * t[4][1]) + sq(t[2][4] * t[3][1]) + sq(t[3][4] * t[2][1]));
        const CL Bm = (L)gm * nt * (sq(s[2][0] * s[3][4]) + sq(s[3][0] * s[2][4]) + sq(s[4][0] * s[2][3]));
        m[0] = (double)mA;
        m[1] = (double)mP;
        m[2] = (double)(std::norm(Bp) + std::norm(Bm));
        m[3] = (double)X.real();
        m[4] = (double)X.imag();
    }
}

// tp_helicity.h -- the five helicity sums of an event (matelems.rs:53-86) from
// its photon momenta, in closed form.
//
// The reference evaluates eight helicity amplitudes from spinor products
// (spinor.rs:31-162) and sums their squares.  Every amplitude is a monomial of
// those products, or a sum of three, so the sums over helicities reduce to
// real and complex polynomials in the momenta and one reciprocal, without the
// spinors' square roots.  With ez = E + Z and c = X + i Y the spinor of a
// photon is (sqrt(ez), c / sqrt(ez)); the beams run along x (evgen.rs:66-69),
// so with h = e_total / 2
//   s(0,k) = -sqrt(h / ez) (ez + c),   s(1,k) = sqrt(h / ez) (ez - c),
//   s(a,b) = (c_a ez_b - c_b ez_a) / sqrt(ez_a ez_b),   t = -conj(s).
// For photon k let N0 = |ez + c|^2, N1 = |ez - c|^2, w = N0 N1, g = ez^2 - c^2
// (|g|^2 = w), and for the pair (a, b) beside it V = c_a ez_b - c_b ez_a,
// D = V^2 and ee = (ez_a ez_b)^2; let Z = (ez_0 ez_1 ez_2)^2, W = w_0 w_1 w_2:
//   sum |A|^2   = (ka/h)^2 / (Z W)    sum_k (N0^2 + N1^2) w ee ee
//   sum |B+|^2  = (kp h)^2 / Z        sum_k (N0^2 + N1^2) |V|^4
//   sum 2 A B+* = -2 ka kp / (Z W)    sum_k w ee [(N0^2 + N1^2) Re T + i (N0^2 - N1^2) Im T],
//                                     T = D conj(g_a g_b)
//   sum |B-|^2  = 2 (km h)^2 / Z      (|sum_k (ez^2 + c^2) D|^2 + 4 |sum_k ez c D|^2)
// where ka, kp, km are (-RAC8) s(0,1) times the couplings (t(0,1) = -s(0,1)).
// The photons enter symmetrically, so their order only moves the rounding.
// The masslessness of the momenta is not used (RAMBO's hold it to a few ulp of
// the conformal map's condition): the sums are the ones of the reference's
// spinors for the same momenta.  Against long double over 4e5 events they are
// within 3.7 eps at p99 and 13.5 eps at most, where the reference's own order
// of operations is within 5.8 and 26.
//
// What bounds it: VALU issue, about 210 f64 instructions an accepted event
// where the amplitudes took 424 (the event loop 32.6 -> 27.5 ms per 1e9 events).
//
// The sums reach the 18th power of the energy, so the caller gives momenta in
// units in which e_total is of order 100 (see energy_unit).
//
// The same source builds for the host (g++), where the tests measure it.
#pragma once

#include "tp_math.h"

namespace tpd {

struct HelicityK { // run constants of the sums above
    double a, p, m, x; // (ka/h)^2, (kp h)^2, 2 (km h)^2, -2 ka kp
};

// p[k] = photon k as (X, Y, Z, E), in any order.
TPM_FN void helicity_sums_closed(const HelicityK &K, const double p[3][4], double m[5])
{
    using tpm::fma_;
    double ez[3], px[3], py[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        ez[k] = p[k][3] + p[k][2];
        px[k] = p[k][0];
        py[k] = p[k][1];
    }
    // A photon exactly along -Z has the spinor (0, sqrt(2E)) (spinor.rs:40-44),
    // the limit ez -> 0 of (ez, sqrt(2 E ez)) / sqrt(ez); one with E below -Z
    // has none (the reference's sqrt is NaN, and so are its sums).
    if (!(ez[0] > 0. && ez[1] > 0. && ez[2] > 0.)) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (ez[k] == 0.) {
                ez[k] = p[k][3] * 0x1.0p-120;
                px[k] = tpm::sqrt_n(2. * p[k][3] * ez[k]);
                py[k] = 0.;
            }
            if (!(ez[k] > 0.))
                ez[k] = __builtin_nan("");
        }
    }
    const double e2[3] = {ez[0] * ez[0], ez[1] * ez[1], ez[2] * ez[2]};
    const double ee[3] = {e2[1] * e2[2], e2[0] * e2[2], e2[0] * e2[1]};
    double W = 1., q[3], t[3], td[3], gr[3], gi[3], sA = 0.;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double a = ez[k] + px[k], b = ez[k] - px[k], y2 = py[k] * py[k];
        const double n0 = fma_(a, a, y2), n1 = fma_(b, b, y2), n12 = n1 * n1;
        const double w = n0 * n1, we = w * ee[k];
        W = k == 0 ? w : W * w;
        q[k] = fma_(n0, n0, n12);               // N0^2 + N1^2
        t[k] = q[k] * we;
        td[k] = fma_(n0, n0, -n12) * we;        // (N0^2 - N1^2) w ee
        sA = k == 0 ? t[k] * ee[k] : fma_(t[k], ee[k], sA);
        gr[k] = fma_(a, b, y2);                 // Re g
        gi[k] = (px[k] + px[k]) * py[k];        // -Im g = Im (ez^2 + c^2)
    }
    double sP = 0., sR = 0., sI = 0., ur = 0., ui = 0., vr = 0., vi = 0.;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int a = k == 0 ? 1 : 0, b = k == 2 ? 1 : 2;
        const double Vr = fma_(px[a], ez[b], -(px[b] * ez[a])), Vi = fma_(py[a], ez[b], -(py[b] * ez[a]));
        const double Vi2 = Vi * Vi, Dr = fma_(Vr, Vr, -Vi2), Dn = fma_(Vr, Vr, Vi2), Di = (Vr + Vr) * Vi;
        const double Gr = fma_(gr[a], gr[b], -(gi[a] * gi[b])), Gi = fma_(gr[a], gi[b], gi[a] * gr[b]); // conj(g_a g_b)
        const double Tr = fma_(Dr, Gr, -(Di * Gi)), Ti = fma_(Dr, Gi, Di * Gr);
        const double hr = fma_(px[k], px[k], e2[k] - py[k] * py[k]), cr = ez[k] * px[k], ci = ez[k] * py[k]; // ez^2 + c^2, ez c
        if (k == 0) { // the first terms start the sums
            sP = (Dn * Dn) * q[k];
            sR = t[k] * Tr;
            sI = td[k] * Ti;
            ur = fma_(hr, Dr, -(gi[k] * Di));
            ui = fma_(hr, Di, gi[k] * Dr);
            vr = fma_(cr, Dr, -(ci * Di));
            vi = fma_(cr, Di, ci * Dr);
        } else {
            sP = fma_(Dn * Dn, q[k], sP);
            sR = fma_(t[k], Tr, sR);
            sI = fma_(td[k], Ti, sI);
            ur = fma_(hr, Dr, fma_(-gi[k], Di, ur));
            ui = fma_(hr, Di, fma_(gi[k], Dr, ui));
            vr = fma_(cr, Dr, fma_(-ci, Di, vr));
            vi = fma_(cr, Di, fma_(ci, Dr, vi));
        }
    }
    const double Z = ee[2] * e2[2], izw = tpm::rcp_n(Z * W), iz = W * izw;
    const double x = K.x * izw;
    m[0] = (K.a * izw) * sA;
    m[1] = (K.p * iz) * sP;
    m[2] = (K.m * iz) * fma_(4., fma_(vr, vr, vi * vi), fma_(ur, ur, ui * ui));
    m[3] = x * sR;
    m[4] = x * sI;
}

// The power of two that takes e_total into [64, 128) (1 for the shipped
// 91.187 GeV): momenta and energies scaled by it keep every bit.
inline double energy_unit(double e_total)
{
    int e = 0;
    (void)std::frexp(e_total, &e); // e_total in [2^(e-1), 2^e)
    return std::ldexp(1., 7 - e < -1000 ? -1000 : 7 - e > 1000 ? 1000 : 7 - e);
}

// The constants for momenta times `unit`, the sums coming out in the caller's
// own units: sum |A|^2 has the dimension of energy^-2, the interference of
// energy^2 and the other two of energy^6, apart from ka^2, ka kp, kp^2, km^2.
inline HelicityK helicity_constants(double e_total, double g_a, double g_bp, double g_bm, double unit)
{
    const double h = e_total / 2., s = 2. * 1.41421356237309504880 * e_total; // (-RAC8) s(0,1)
    const double ka = s * g_a, kp = s * g_bp, km = s * g_bm, u2 = unit * unit, u6 = u2 * u2 * u2;
    return HelicityK{(ka / h) * (ka / h) * u2, (kp * h) * (kp * h) / u6, 2. * ((km * h) * (km * h)) / u6,
                     -2. * (ka * kp) / u2};
}

} // namespace tpd

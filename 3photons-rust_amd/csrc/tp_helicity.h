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

// The sums and their derivatives.  With zeta = c / ez the sums separate: for
// photon k let n0 = |1 + zeta|^2, n1 = |1 - zeta|^2, s = |zeta|^2,
//   u = ez^2 (n0^2 + n1^2) = ez^2 (2 (1 + s)^2 + 8 Re(zeta)^2),
//   v = ez^2 (n0^2 - n1^2) = 8 ez^2 (1 + s) Re(zeta),
//   rho = 1 / (ez^2 n0 n1),  f = 1 / (1 - zeta^2),
// and for the pair (a, b) beside it d = zeta_a - zeta_b, S = ez_a ez_b |d|^2 and
// tau = d^2 f_a f_b; with Z as above
//   sum |A|^2  = K.a sum_k u rho_a rho_b,     sum |B+|^2 = K.p sum_k u S^2,
//   sum 2 A B* = K.x sum_k (u Re tau + i v Im tau),
//   sum |B-|^2 = K.m Z (|sum_k (1 + zeta^2) d^2|^2 + 4 |sum_k zeta d^2|^2),
// where tau and the two sums of the last line are analytic in the zetas.  The
// derivatives by (ez, Re zeta, Im zeta) go over to (X, Y, ez) at the end; by
// E and by Z are the one by ez.
//
// m[5]: the sums; g[c][k] = d m_c / d (X, Y, ez) of photon k.  `along`: bit k is
// set for a photon with the spinor (0, sqrt(2 E)), which depends on E alone; its
// X and Y derivatives are 0 and g[c][k][2] is the one by E (a photon with E
// below -Z counts as one too, and its sums and derivatives are NaN).  A photon
// without energy (RAMBO's from u1 u2 = 1, which given points may have and only
// cuts that are off let pass) has the spinor (0, 0), a factor of every B and a
// divisor of A: the sums of the B are 0 (bit 3), all else NaN.
TPM_FN void helicity_gradients(const HelicityK &K, const double p[3][4], double m[5], double g[5][3][3], int &along)
{
    using tpm::fma_;
    double ez[3], px[3], py[3];
    along = 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        ez[k] = p[k][3] + p[k][2];
        px[k] = p[k][0];
        py[k] = p[k][1];
    }
    if (!(ez[0] > 0. && ez[1] > 0. && ez[2] > 0.)) { // as in helicity_sums_closed
        bool spinors = true;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if (!(ez[k] > 0.))
                along |= 1 << k;
            if (ez[k] == 0. && p[k][3] == 0.)
                along |= 8;
            spinors = spinors && ez[k] >= 0.;
            if (ez[k] == 0.) {
                ez[k] = p[k][3] * 0x1.0p-120;
                px[k] = tpm::sqrt_n(2. * p[k][3] * ez[k]);
                py[k] = 0.;
            }
            if (!(ez[k] > 0.))
                ez[k] = __builtin_nan("");
        }
        along = spinors ? along : along & 7;
    }
    double iz[3], zr[3], zi[3], u[3], v[3], rho[3], fr[3], fi[3], Gr[3], Gi[3], ur[3], ui[3], vr[3], vi[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        iz[k] = tpm::rcp_n(ez[k]);
        zr[k] = px[k] * iz[k];
        zr[k] = fma_(fma_(-zr[k], ez[k], px[k]), iz[k], zr[k]);
        zi[k] = py[k] * iz[k];
        zi[k] = fma_(fma_(-zi[k], ez[k], py[k]), iz[k], zi[k]);
        const double a = 1. + zr[k], b = 1. - zr[k], y2 = zi[k] * zi[k], x2 = zr[k] * zr[k];
        const double n0 = fma_(a, a, y2), n1 = fma_(b, b, y2), in = tpm::rcp_n(n0 * n1);
        fr[k] = fma_(a, b, y2) * in;
        fi[k] = ((zr[k] + zr[k]) * zi[k]) * in;
        Gr[k] = fma_(zr[k], fr[k], -(zi[k] * fi[k])); // zeta f: d f / d zeta = 2 zeta f^2
        Gi[k] = fma_(zr[k], fi[k], zi[k] * fr[k]);
        rho[k] = (iz[k] * iz[k]) * in;
        const double s = x2 + y2, h = 1. + s, e2 = ez[k] * ez[k], e8 = 8. * e2;
        u[k] = fma_(e8, x2, (2. * e2) * (h * h));
        v[k] = (e8 * h) * zr[k];
        ur[k] = (e8 * (3. + s)) * zr[k];
        ui[k] = (e8 * h) * zi[k];
        vr[k] = e8 * fma_(2., x2, h);
        vi[k] = (2. * e8) * (zr[k] * zi[k]);
    }
    // derivatives by (Re zeta, Im zeta), and ez times the one by ez
    double wr[5][3], wi[5][3], we[5][3];
    double dr[3], di[3], Dr[3], Di[3];
    // Pair k is (a, b) = (1, 2), (0, 2), (0, 1): photon j is its first member if
    // j < k or (j, k) = (1, 0), else its second, where d counts negative.
    double tr[3], ti[3], Pr = 0., Pi = 0., Tr = 0., Ti = 0.;
    double tAr[3][3], tAi[3][3]; // d tau_k / d zeta_j
    double cS[3];                // 2 K.p u S ez_a ez_b of the pair, twice
    m[1] = 0.;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int a = k == 0 ? 1 : 0, b = k == 2 ? 1 : 2;
        dr[k] = zr[a] - zr[b];
        di[k] = zi[a] - zi[b];
        const double di2 = di[k] * di[k], ab = ez[a] * ez[b];
        Dr[k] = fma_(dr[k], dr[k], -di2);
        Di[k] = (dr[k] + dr[k]) * di[k];
        const double S = ab * fma_(dr[k], dr[k], di2), KS = K.p * S;
        cS[k] = (4. * u[k]) * (KS * ab);
        const double aS = KS * S;
        wr[1][k] = aS * ur[k];
        wi[1][k] = aS * ui[k];
        m[1] = fma_(aS, u[k], m[1]);
        const double hr = fma_(fr[a], fr[b], -(fi[a] * fi[b])), hi = fma_(fr[a], fi[b], fi[a] * fr[b]);
        tr[k] = fma_(Dr[k], hr, -(Di[k] * hi));
        ti[k] = fma_(Dr[k], hi, Di[k] * hr);
        const double d2r = dr[k] + dr[k], d2i = di[k] + di[k], t2r = tr[k] + tr[k], t2i = ti[k] + ti[k];
        const double er = fma_(d2r, hr, -(d2i * hi)), ei = fma_(d2r, hi, d2i * hr);
        tAr[k][a] = fma_(t2r, Gr[a], fma_(-t2i, Gi[a], er));
        tAi[k][a] = fma_(t2r, Gi[a], fma_(t2i, Gr[a], ei));
        tAr[k][b] = fma_(t2r, Gr[b], fma_(-t2i, Gi[b], -er));
        tAi[k][b] = fma_(t2r, Gi[b], fma_(t2i, Gr[b], -ei));
        Tr = fma_(zr[k], Dr[k], fma_(-zi[k], Di[k], Tr));
        Ti = fma_(zr[k], Di[k], fma_(zi[k], Dr[k], Ti));
        const double qr = fma_(zr[k], zr[k], fma_(-zi[k], zi[k], 1.)), qi = (zr[k] + zr[k]) * zi[k];
        Pr = fma_(qr, Dr[k], fma_(-qi, Di[k], Pr));
        Pi = fma_(qr, Di[k], fma_(qi, Dr[k], Pi));
    }
    // sum |A|^2 and the interference
    double A[3], AU[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int a = k == 0 ? 1 : 0, b = k == 2 ? 1 : 2;
        A[k] = (K.a * rho[a]) * rho[b];
        AU[k] = A[k] * u[k];
    }
    m[0] = (AU[0] + AU[1]) + AU[2];
    m[3] = K.x * fma_(u[0], tr[0], fma_(u[1], tr[1], u[2] * tr[2]));
    m[4] = K.x * fma_(v[0], ti[0], fma_(v[1], ti[1], v[2] * ti[2]));
    const double Z = (ez[0] * ez[1]) * ez[2], KZ = (K.m * Z) * Z;
    m[2] = KZ * fma_(4., fma_(Tr, Tr, Ti * Ti), fma_(Pr, Pr, Pi * Pi));
    const double K2 = KZ + KZ, Kx2 = K.x + K.x;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int a = k == 0 ? 1 : 0, b = k == 2 ? 1 : 2;
        const double bk = 4. * (AU[a] + AU[b]); // 4 rho d / d rho
        wr[0][k] = fma_(bk, Gr[k], A[k] * ur[k]);
        wi[0][k] = fma_(-bk, Gi[k], A[k] * ui[k]);
        we[0][k] = fma_(-0.5, bk, AU[k] + AU[k]);
        // pair a is (k, b) or (b, k), pair b is (k, a) or (a, k)
        const double sa = k < b ? cS[a] : -cS[a], sb = k < a ? cS[b] : -cS[b];
        wr[1][k] = fma_(sa, dr[a], fma_(sb, dr[b], wr[1][k]));
        wi[1][k] = fma_(sa, di[a], fma_(sb, di[b], wi[1][k]));
        we[1][k] = m[1] + m[1];
        const double Rr = fma_(u[a], tAr[a][k], u[b] * tAr[b][k]), Ri = fma_(u[a], tAi[a][k], u[b] * tAi[b][k]);
        const double Ir = fma_(v[a], tAr[a][k], v[b] * tAr[b][k]), Ii = fma_(v[a], tAi[a][k], v[b] * tAi[b][k]);
        wr[3][k] = K.x * fma_(ur[k], tr[k], Rr);
        wi[3][k] = K.x * fma_(ui[k], tr[k], -Ri);
        we[3][k] = Kx2 * (u[k] * tr[k]);
        wr[4][k] = K.x * fma_(vr[k], ti[k], Ii);
        wi[4][k] = K.x * fma_(vi[k], ti[k], Ir);
        we[4][k] = Kx2 * (v[k] * ti[k]);
        // d/d zeta_k of sum zeta d^2 and, halved, of sum (1 + zeta^2) d^2
        const double ga = k < b ? 1. : -1., gb = k < a ? 1. : -1.;
        const double Yar = fma_(zr[a], dr[a], -(zi[a] * di[a])), Yai = fma_(zr[a], di[a], zi[a] * dr[a]);
        const double Ybr = fma_(zr[b], dr[b], -(zi[b] * di[b])), Ybi = fma_(zr[b], di[b], zi[b] * dr[b]);
        const double T1r = fma_(2., fma_(ga, Yar, gb * Ybr), Dr[k]), T1i = fma_(2., fma_(ga, Yai, gb * Ybi), Di[k]);
        const double Wr = fma_(ga, fma_(zr[a], Yar, fma_(-zi[a], Yai, dr[a])), gb * fma_(zr[b], Ybr, fma_(-zi[b], Ybi, dr[b])));
        const double Wi = fma_(ga, fma_(zr[a], Yai, fma_(zi[a], Yar, di[a])), gb * fma_(zr[b], Ybi, fma_(zi[b], Ybr, di[b])));
        const double P1r = fma_(zr[k], Dr[k], fma_(-zi[k], Di[k], Wr)), P1i = fma_(zr[k], Di[k], fma_(zi[k], Dr[k], Wi));
        // 2 conj(P) P1 + 4 conj(T) T1
        const double hr = fma_(4., fma_(Tr, T1r, Ti * T1i), 2. * fma_(Pr, P1r, Pi * P1i));
        const double hi = fma_(4., fma_(Tr, T1i, -(Ti * T1r)), 2. * fma_(Pr, P1i, -(Pi * P1r)));
        wr[2][k] = K2 * hr;
        wi[2][k] = -(K2 * hi);
        we[2][k] = m[2] + m[2];
    }
#pragma unroll
    for (int c = 0; c < 5; ++c)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            g[c][k][0] = wr[c][k] * iz[k];
            g[c][k][1] = wi[c][k] * iz[k];
            g[c][k][2] = fma_(-zr[k], wr[c][k], fma_(-zi[k], wi[c][k], we[c][k])) * iz[k];
        }
    if (along) {
        if (along & 8)
            m[1] = m[2] = 0.;
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (along >> k & 1) // X = sqrt(ez) sqrt(2 E): d/dE = d/dX ez / X
#pragma unroll
                for (int c = 0; c < 5; ++c) {
                    g[c][k][2] = g[c][k][0] / zr[k];
                    g[c][k][0] = g[c][k][1] = 0.;
                }
    }
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

// Pointwise pieces of the discrete adjoint (cav3d_rhs_vjp): the gradient of
// one face's inviscid flux, one face's viscous flux and one cell's
// properties with respect to their inputs.  Each is the physics of phys.hpp
// run backwards by hand: the forward values once, then every operation's
// transpose in reverse, following the branches, clamps and min/max
// selections the forward values took (at ties as phys.hpp's mx / mn choose,
// which is also what the dual numbers do).  A gradient costs two to three
// evaluations whatever its number of inputs, where forward-mode passes of two
// lanes cost one evaluation and a half for every two inputs.  Roe-M and
// AUSMPW+, which no default uses, keep the dual passes (Dn<W>).  Host and
// device: the host build is checked against finite differences and against
// dual-number passes of the same physics.
#pragma once
#include "phys.hpp"

namespace cav {

constexpr int NSLOT = 38;   // the reference's face stencil, Fortran numbering 1..38

// Gradient of a scalar function of n inputs by dual passes of W lanes:
// x(q) is the value of input q; f(in, base) evaluates phi reading input q as
// in(q), which carries lane q - base when that lies in 0..W-1; gx[q] =
// d phi / d x[q].  The inputs are seeded where they are read (no array of
// duals is kept), which keeps the private memory per lane small.
template <int W, class X, class F>
HD void dn_grad(int n, X x, F f, double *gx)
{
    for (int base = 0; base < n; base += W) {
        auto in = [&](int q) -> Dn<W> { return Dn<W>::seed(x(q), q - base); };
        const Dn<W> phi = f(in, base);
        for (int l = 0; l < W; l++) if (base + l < n) gx[base + l] = phi.d[l];
    }
}

// muscl_clamps with the origin of every face value: 0 the reconstruction,
// 1 the cell, 2 the pressure floor (a constant in absolute pressure)
__host__ __device__ inline void clamps_src(int npv, double pref, const double *c9, const double *c10, double *xl, double *xr,
                           int *ol, int *orr)
{
    for (int n = 0; n < NPV; n++) ol[n] = orr[n] = 0;
    const double fl = -pref + 10.0;
    if (!(xl[0] > fl)) { xl[0] = fl; ol[0] = 2; }
    if (!(xr[0] > fl)) { xr[0] = fl; orr[0] = 2; }
    if ((xl[5] < 0.0) || (xl[5] > 1.0)) { xl[5] = c9[5]; ol[5] = 1; }
    if ((xr[5] < 0.0) || (xr[5] > 1.0)) { xr[5] = c10[5]; orr[5] = 1; }
    if ((xl[6] < 0.0) || (xl[6] > 1.0)) { xl[6] = c9[6]; ol[6] = 1; }
    if ((xr[6] < 0.0) || (xr[6] > 1.0)) { xr[6] = c10[6]; orr[6] = 1; }
    if ((xl[5] + xl[6]) > 1.0) { xl[5] = c9[5]; xl[6] = c9[6]; ol[5] = ol[6] = 1; }
    if ((xr[5] + xr[6]) > 1.0) { xr[5] = c10[5]; xr[6] = c10[6]; orr[5] = orr[6] = 1; }
    if (npv > 7) {
        if ((xl[7] < 0.0) && (c9[7] > 0.0)) { xl[7] = c9[7]; ol[7] = 1; }
        if ((xr[7] < 0.0) && (c10[7] > 0.0)) { xr[7] = c10[7]; orr[7] = 1; }
        if ((xl[8] < 0.0) && (c9[8] > 0.0)) { xl[8] = c9[8]; ol[8] = 1; }
        if ((xr[8] < 0.0) && (c10[8] > 0.0)) { xr[8] = c10[8]; orr[8] = 1; }
    }
}

// ------------------------------------------------------------ phases
// A phase's six E2 values with their derivatives with respect to p and T (the
// derivatives of the formulas as phys.hpp evaluates them, folded constants
// included): v = {rho, h, drho/dp, drho/dT, dh/dp, dh/dT}.
struct E2x { double v[6], p[6], t[6]; };
enum { EX_RHO = 0, EX_H, EX_RP, EX_RT, EX_HP, EX_HT };

// from the sums of the dimensionless Gibbs function: G = dg/dpi and its
// derivatives with respect to pi and tau, gt = dg/dtau and its tau
// derivatives; pi = kp p, tau = const / t, and the E2 constants
HD void e2x_fill(E2x &e, double G, double Gp, double Gt, double Gpp, double Gpt, double Gtt, double gt, double gtt, double gttt,
                 double tau, double t, double kp, double crho, double ch, double crp, double crt1, double crt2, double chp)
{
    const double i1 = 1.0 / G, i2 = i1 * i1, i3 = i2 * i1, t2 = tau * tau, t3 = t2 * tau;
    // values and their derivatives with respect to pi (_p) and tau (_t)
    const double rho = crho * tau * i1, rho_p = -(crho * tau * i2 * Gp), rho_t = crho * (i1 - tau * i2 * Gt);
    const double h_p = ch * Gt, h_t = ch * gtt;
    const double rp = -(Gp * crp * tau * i2);
    const double rp_p = -(crp * tau * (Gpp * i2 - 2.0 * Gp * Gp * i3));
    const double rp_t = -(crp * (Gpt * tau * i2 + Gp * i2 - 2.0 * Gp * tau * i3 * Gt));
    const double rt = -(rho * crt1 * tau) + crt2 * Gt * t3 * i2;
    const double rt_p = -(rho_p * crt1 * tau) + crt2 * t3 * (Gpt * i2 - 2.0 * Gt * i3 * Gp);
    const double rt_t = -(crt1 * (rho_t * tau + rho)) + crt2 * (Gtt * t3 * i2 + 3.0 * Gt * t2 * i2 - 2.0 * Gt * t3 * i3 * Gt);
    const double ht = -(461.526 * t2 * gtt), ht_p = -(461.526 * t2 * Gtt), ht_t = -(461.526 * (2.0 * tau * gtt + t2 * gttt));
    const double kt = -tau / t;
    e.v[EX_RHO] = rho; e.p[EX_RHO] = rho_p * kp; e.t[EX_RHO] = rho_t * kt;
    e.v[EX_H] = ch * gt; e.p[EX_H] = h_p * kp; e.t[EX_H] = h_t * kt;
    e.v[EX_RP] = rp; e.p[EX_RP] = rp_p * kp; e.t[EX_RP] = rp_t * kt;
    e.v[EX_RT] = rt; e.p[EX_RT] = rt_p * kp; e.t[EX_RT] = rt_t * kt;
    e.v[EX_HP] = chp * Gt; e.p[EX_HP] = chp * Gpt * kp; e.t[EX_HP] = chp * Gtt * kt;
    e.v[EX_HT] = ht; e.p[EX_HT] = ht_p * kp; e.t[EX_HT] = ht_t * kt;
}

// Region 1 (liquid<R>) to third order in the Gibbs function
HD void liquid_x(double p, double t, E2x &e)
{
    const double kp = 0.00000006049607;
    const double pi = p * kp, tau = 1386.0 / t, q = 7.1 - pi, w = tau - 1.222;
    const double pi1 = 1.0 / q, tau1 = 1.0 / w;
    double gt = 0, gp = 0, gpp = 0, gtt = 0, gpt = 0, gppp = 0, gppt = 0, gptt = 0, gttt = 0;
#pragma unroll
    for (int k = 0; k < 34; k++) {
        const int I = R1C[k].i, J = R1C[k].j;
        const double g = R1C[k].n * powi(q, I) * powi(w, J);
        const double g1 = J * g * tau1, g2 = -(I * g * pi1), g3 = -((I - 1) * g2 * pi1), g4 = (J - 1) * g1 * tau1, g5 = J * g2 * tau1;
        gt += g1; gp += g2; gpp += g3; gtt += g4; gpt += g5;
        gppp -= (I - 2) * g3 * pi1;
        gppt += J * g3 * tau1;
        gptt += (J - 1) * g5 * tau1;
        gttt += (J - 2) * g4 * tau1;
    }
    e2x_fill(e, gp, gpp, gpt, gppp, gppt, gptt, gt, gtt, gttt, tau, t, kp, C_RHO1, 639675.036, 1.5632937721834122e-6,
             7.215007215007215e-4, C_RT1, C_HP1);
}

// Region 2 with the metastable branch (vapour<R>)
HD void vapour_x(double p, double t, double psat, E2x &e)
{
    const double kp = 1.0e-6;
    const double pi = p * kp, tau = 540.0 / t, w = tau - 0.5;
    const double pi1 = 1.0e6 / p, tau1 = 1.0 / tau, tau2 = 1.0 / w;
    const bool meta = p > psat;
    double gt = 0, gtt = 0, gttt = 0, gp = 0, gpp = 0, gpt = 0, gppp = 0, gppt = 0, gptt = 0;
#pragma unroll
    for (int k = 0; k < 9; k++) {
        const int J = R2J0[k];
        const double n = (meta && k < 2) ? R2MN0[k < 2 ? k : 0] : R2N0[k];
        const double g0 = n * powi(tau, J), g1 = J * g0 * tau1, g2 = (J - 1) * g1 * tau1;
        gt += g1; gtt += g2;
        gttt += (J - 2) * g2 * tau1;
    }
    auto term = [&](const IJN c) {
        const double g = c.n * powi(pi, c.i) * powi(w, c.j);
        const double g1 = c.j * g * tau2, g2 = c.i * g * pi1, g3 = (c.i - 1) * g2 * pi1, g4 = (c.j - 1) * g1 * tau2, g5 = c.j * g2 * tau2;
        gt += g1; gp += g2; gpp += g3; gtt += g4; gpt += g5;
        gppp += (c.i - 2) * g3 * pi1;
        gppt += c.j * g3 * tau2;
        gptt += (c.j - 1) * g5 * tau2;
        gttt += (c.j - 2) * g4 * tau2;
    };
    if (meta) {
#pragma unroll
        for (int k = 0; k < 13; k++) term(R2MC[k]);
    } else {
#pragma unroll
        for (int k = 0; k < 43; k++) term(R2C[k]);
    }
    const double q2 = pi1 * pi1;
    e2x_fill(e, pi1 + gp, gpp - q2, gpt, gppp + 2.0 * q2 * pi1, gppt, gptt, gt, gtt, gttt, tau, t, kp, 4.01245401527075799,
             249224.04, 4.01245401527075799e-6, C_RT2A, C_RT2B, 0.24922404);
}

HD void gas_x(double p, double t, E2x &e)
{
    const double r1 = 0.00348383500557, tau = 1.0 / t;
    const double rp = r1 * tau, rt = -(p * r1 * (tau * tau));
    e.v[EX_RHO] = p * r1 * tau; e.p[EX_RHO] = rp; e.t[EX_RHO] = rt;
    e.v[EX_H] = 1004.64 * t; e.p[EX_H] = 0.0; e.t[EX_H] = 1004.64;
    e.v[EX_RP] = rp; e.p[EX_RP] = 0.0; e.t[EX_RP] = -(rp * tau);
    e.v[EX_RT] = rt; e.p[EX_RT] = -(r1 * (tau * tau)); e.t[EX_RT] = -2.0 * rt * tau;
    e.v[EX_HP] = e.p[EX_HP] = e.t[EX_HP] = 0.0;
    e.v[EX_HT] = 1004.64; e.p[EX_HT] = e.t[EX_HT] = 0.0;
}

// Gradient with respect to (p, T, y1, y2) of sum_m w[m] d[m] over the mixture's
// thermodynamic properties (mixture_eos), from the phases' E2x.  The
// mixture sums are run forward; then the seeds go back through them to the
// phases' specific volumes, E2 values and mass fractions.
HD void mixture_back(const E2x &l, const E2x &v, const E2x &g, double y1, double y2, const double *w, double *gx)
{
    const double y[3] = {1.0 - y1 - y2, y1, y2};
    const E2x *e[3] = {&l, &v, &g};
    double i[3], S = 0, srp = 0, srt = 0, hp = 0, ht = 0;
    for (int k = 0; k < 3; k++) {
        i[k] = 1.0 / e[k]->v[EX_RHO];
        S += y[k] * i[k];
        srp += y[k] * (i[k] * i[k]) * e[k]->v[EX_RP];
        srt += y[k] * (i[k] * i[k]) * e[k]->v[EX_RT];
        hp += y[k] * e[k]->v[EX_HP];
        ht += y[k] * e[k]->v[EX_HT];
    }
    const double rho = 1.0 / S, r2 = rho * rho, rp = r2 * srp, rt = r2 * srt;
    const double den = rho * rp * ht + rt * (1.0 - rho * hp);
    // bars of rho, r2's own appearances, the sums and the phase values
    double rhob = w[D_RHO], rpb = w[D_RP], rtb = w[D_RT], hpb = w[D_HP], htb = w[D_HT], r2b = 0.0;
    double ib[3] = {0, 0, 0}, yb[3] = {0, 0, 0}, eb[3][6] = {};
    if (w[D_C2] != 0.0) {
        const double c2 = rho * ht / den;
        if (!(c2 <= 0.0)) {
            const double nb = w[D_C2] / den, db = -(nb * c2);
            rhob += nb * ht + db * (rp * ht - rt * hp);
            htb += nb * rho + db * rho * rp;
            rpb += db * rho * ht;
            rtb += db * (1.0 - rho * hp);
            hpb -= db * rt * rho;
        } else {       // the phase-weighted fallback of mixture_eos
            double cs = 0.0, c[3];
            for (int k = 0; k < 3; k++) {
                const double *q = e[k]->v;
                c[k] = (q[EX_RHO] * q[EX_RP] * q[EX_HT] + q[EX_RT] * (1.0 - q[EX_RHO] * q[EX_HP])) / (q[EX_RHO] * q[EX_HT]);
                cs += y[k] * c[k] * (i[k] * i[k]);
            }
            const double f = 1.0 / (r2 * cs), fb = -(w[D_C2] * f * f);
            r2b += fb * cs;
            for (int k = 0; k < 3; k++) {
                const double *q = e[k]->v;
                const double sb = fb * r2;
                yb[k] += sb * c[k] * (i[k] * i[k]);
                ib[k] += sb * y[k] * c[k] * 2.0 * i[k];
                // c = rp + rt / (rho ht) - rt hp / ht
                const double cb = sb * y[k] * (i[k] * i[k]), rh = 1.0 / (q[EX_RHO] * q[EX_HT]);
                eb[k][EX_RP] += cb;
                eb[k][EX_RT] += cb * (1.0 - q[EX_RHO] * q[EX_HP]) * rh;
                eb[k][EX_RHO] -= cb * q[EX_RT] * rh / q[EX_RHO];
                eb[k][EX_HP] -= cb * q[EX_RT] / q[EX_HT];
                eb[k][EX_HT] -= cb * q[EX_RT] * (1.0 - q[EX_RHO] * q[EX_HP]) * rh / q[EX_HT];
            }
        }
    }
    // rho_y1 = r2 (il - iv), rho_y2 = r2 (il - ig)
    r2b += w[D_RY1] * (i[0] - i[1]) + w[D_RY2] * (i[0] - i[2]) + rpb * srp + rtb * srt;
    ib[0] += r2 * (w[D_RY1] + w[D_RY2]);
    ib[1] -= r2 * w[D_RY1];
    ib[2] -= r2 * w[D_RY2];
    rhob += 2.0 * rho * r2b;
    const double Sb = -(rhob * r2), srpb = rpb * r2, srtb = rtb * r2, hb = w[D_H];
    // h_y1 = hv - hl, h_y2 = hg - hl
    const double hyb[3] = {-(w[D_HY1] + w[D_HY2]), w[D_HY1], w[D_HY2]};
    double pb = 0.0, tb = 0.0;
    for (int k = 0; k < 3; k++) {
        const double *q = e[k]->v, ii = i[k] * i[k];
        yb[k] += Sb * i[k] + srpb * ii * q[EX_RP] + srtb * ii * q[EX_RT] + hpb * q[EX_HP] + htb * q[EX_HT] + hb * q[EX_H];
        ib[k] += y[k] * (Sb + 2.0 * i[k] * (srpb * q[EX_RP] + srtb * q[EX_RT]));
        eb[k][EX_RHO] -= ib[k] * ii;
        eb[k][EX_H] += hb * y[k] + hyb[k];
        eb[k][EX_RP] += srpb * y[k] * ii;
        eb[k][EX_RT] += srtb * y[k] * ii;
        eb[k][EX_HP] += hpb * y[k];
        eb[k][EX_HT] += htb * y[k];
        for (int m = 0; m < 6; m++) { pb += eb[k][m] * e[k]->p[m]; tb += eb[k][m] * e[k]->t[m]; }
    }
    gx[0] = pb; gx[1] = tb; gx[2] = yb[1] - yb[0]; gx[3] = yb[2] - yb[0];
}

HD void phases_x(double p, double t, E2x &l, E2x &v, E2x &g)
{
    liquid_x(p, t, l);
    vapour_x(p, t, sat_p(t), v);
    gas_x(p, t, g);
}

// gradient of c^2 (face_c2, with both phases kept: the mass fractions are inputs)
HD void c2_back(double p, double t, double y1, double y2, double c2b, double *gx)
{
    E2x l, v, g;
    phases_x(p, t, l, v, g);
    double w[ND];
    for (int m = 0; m < ND; m++) w[m] = 0.0;
    w[D_C2] = 1.0;         // (as the flux cores' slopes: formed before the bar is applied)
    mixture_back(l, v, g, y1, y2, w, gx);
    for (int q = 0; q < 4; q++) gx[q] *= c2b;
}

// mu and kappa of a water phase (iaps85) back to t and the phase density
HD void iaps85_back(double t, double rho, double mub, double kapb, double &tb, double &rhob, double &mu, double &kap)
{
    const double tt = t * 0.00154495032985, tt1 = 647.27 / t, a = tt1 - 1.0;
    const double rl = mn(1332.4, rho), rc = mx(1.0e-3, rl), rr = rc * 0.00314699949333, b = rr - 1.0;
    const double rr_r = (rho < 1332.4 && rl > 1.0e-3) ? 0.00314699949333 : 0.0;     // mn, mx as the forward pass takes them
    const double tt_t = 0.00154495032985, tt1_t = -tt1 / t;
    const double sq = sqrt(tt);
    double pa[6], pb[7];
    pa[0] = pb[0] = 1.0;
    for (int k = 1; k < 6; k++) pa[k] = pa[k - 1] * a;
    for (int k = 1; k < 7; k++) pb[k] = pb[k - 1] * b;
    {
        const double den = TPH[0] + TPH[1] * tt1 + TPH[2] * (tt1 * tt1) + TPH[3] * (tt1 * tt1 * tt1);
        const double den_1 = TPH[1] + 2.0 * TPH[2] * tt1 + 3.0 * TPH[3] * (tt1 * tt1);
        double s = 0, sa = 0, sb = 0;
#pragma unroll
        for (int k = 0; k <= 5; k++)
#pragma unroll
            for (int j = 0; j <= 6; j++) {
                const double c = TPHH[k][j];
                s += c * pa[k] * pb[j];
                if (k > 0) sa += c * k * pa[k > 0 ? k - 1 : 0] * pb[j];
                if (j > 0) sb += c * j * pa[k] * pb[j > 0 ? j - 1 : 0];
            }
        const double m0 = sq / den, m1 = exp(rr * s);
        mu = 55.071e-6 * m0 * m1;
        // mu = const sqrt(tt) / den(tt1) exp(rr s(tt1, rr))
        const double l_t = 0.5 / tt * tt_t - den_1 / den * tt1_t + rr * sa * tt1_t;
        const double l_r = (s + rr * sb) * rr_r;
        tb += mub * mu * l_t;
        rhob += mub * mu * l_r;
    }
    {
        const double den = TPL[0] + TPL[1] * tt1 + TPL[2] * (tt1 * tt1) + TPL[3] * (tt1 * tt1 * tt1);
        const double den_1 = TPL[1] + 2.0 * TPL[2] * tt1 + 3.0 * TPL[3] * (tt1 * tt1);
        double s = 0, sa = 0, sb = 0;
#pragma unroll
        for (int k = 0; k <= 4; k++)
#pragma unroll
            for (int j = 0; j <= 5; j++) {
                const double c = TPLL[k][j];
                s += c * pa[k] * pb[j];
                if (k > 0) sa += c * k * pa[k > 0 ? k - 1 : 0] * pb[j];
                if (j > 0) sb += c * j * pa[k] * pb[j > 0 ? j - 1 : 0];
            }
        const double l0 = sq / den, l1 = exp(rr * s);
        kap = 0.4945 * (l0 * l1);
        const double l_t = 0.5 / tt * tt_t - den_1 / den * tt1_t + rr * sa * tt1_t;
        const double l_r = (s + rr * sb) * rr_r;
        tb += kapb * kap * l_t;
        rhob += kapb * kap * l_r;
    }
}

// property bars of one cell back to (p, T, y1, y2) through its EOS
__host__ __device__ __attribute__((always_inline)) inline void eos_adj(bool prop, const double *x4, const double *dcb, double *gx)
{
    const double t = x4[1], y1 = x4[2], y2 = x4[3];
    E2x l, v, g;
    phases_x(x4[0], t, l, v, g);
    double w[ND];
    for (int m = 0; m < ND; m++) w[m] = dcb[m];
    double pb = 0.0, tb = 0.0, y1b = 0.0, y2b = 0.0;
    if (prop && (dcb[D_MU] != 0.0 || dcb[D_KAP] != 0.0)) {
        // mu = rho (ml yl il + mv y1 iv + mg y2 ig), kappa alike
        const double yl = 1.0 - y1 - y2, il = 1.0 / l.v[EX_RHO], iv = 1.0 / v.v[EX_RHO], ig = 1.0 / g.v[EX_RHO];
        const double rho = 1.0 / (yl * il + y1 * iv + y2 * ig), mub = dcb[D_MU], kapb = dcb[D_KAP];
        double ml, kl, mv, kv, tl = 0.0, rl = 0.0, tv = 0.0, rv = 0.0;
        iaps85_back(t, l.v[EX_RHO], mub * rho * yl * il, kapb * rho * yl * il, tl, rl, ml, kl);
        iaps85_back(t, v.v[EX_RHO], mub * rho * y1 * iv, kapb * rho * y1 * iv, tv, rv, mv, kv);
        const double pw = pow(t / 273.11, 1.5), mg = 1.716e-5 * pw * 383.67 / (t + 110.56), kg = 1395.333333 * mg;
        const double mg_t = mg * (1.5 / t - 1.0 / (t + 110.56));
        const double bl = mub * ml + kapb * kl, bv = mub * mv + kapb * kv, bg = mub * mg + kapb * kg;
        w[D_RHO] += bl * yl * il + bv * y1 * iv + bg * y2 * ig;
        y1b = rho * (bv * iv - bl * il);
        y2b = rho * (bg * ig - bl * il);
        // the specific volumes' own share: d il = -il^2 d rho_l
        rl -= rho * bl * yl * il * il;
        rv -= rho * bv * y1 * iv * iv;
        const double rg = -(rho * bg * y2 * ig * ig);
        pb = rl * l.p[EX_RHO] + rv * v.p[EX_RHO] + rg * g.p[EX_RHO];
        tb = tl + tv + rl * l.t[EX_RHO] + rv * v.t[EX_RHO] + rg * g.t[EX_RHO]
           + rho * y2 * ig * (mub + kapb * 1395.333333) * mg_t;
    }
    mixture_back(l, v, g, y1, y2, w, gx);
    gx[0] += pb; gx[1] += tb; gx[2] += y1b; gx[3] += y2b;
}

// ------------------------------------------------------------ reconstruction
// The bars of limiter(nlim, m, s)'s r, r1, r2 and alp from its own bar phib.
// The slopes are selected as values (branches that add to one bar or another
// become a store through a selected pointer: four bars in scratch memory
// and a round trip to it in every reconstruction).
struct LimBar { double r, r1, r2, a; };
HD LimBar limiter_back(int nlim, const LimState<double> &m, int s, double phib)
{
    const double r = m.r[s], a = m.alp[s];
    LimBar o{0.0, 0.0, 0.0, 0.0};
    // max(0, min(a, a r, c)), c's slopes (cr, c1, c2) with respect to r, r1, r2
    auto low3 = [&](double c, double cr, double c1, double c2) {
        const double ar = a * r, t = ar < a ? ar : a, v = c < t ? c : t;
        const bool on = v > 0.0, isc = on && c < t, isr = on && !(c < t) && ar < a, isa = on && !(c < t) && !(ar < a);
        o.r = isc ? phib * cr : isr ? phib * a : 0.0;
        o.r1 = isc ? phib * c1 : 0.0;
        o.r2 = isc ? phib * c2 : 0.0;
        o.a = isr ? phib * r : isa ? phib : 0.0;
    };
    // max(0, min(c r, 1), min(r, c)), c's slopes cr and ca with respect to r and a
    auto high2 = [&](double c, double cr, double ca) {
        const double q = c * r, i1 = 1.0 < q ? 1.0 : q, t = i1 > 0.0 ? i1 : 0.0, u = c < r ? c : r;
        const bool up = u > t, isc = up && c < r, isr = up && !(c < r), isq = !up && i1 > 0.0 && !(1.0 < q);
        o.r = isc ? phib * cr : isr ? phib : isq ? phib * (c + cr * r) : 0.0;
        o.a = isc ? phib * ca : isq ? phib * ca * r : 0.0;
    };
    const double ic5 = (-(2.0 * m.r1[s]) + 11.0 + 24.0 * r - 3.0 * m.r2[s]) / 30.0;
    switch (nlim) {
    case 1: o.r = r < 1.0 && r > 0.0 ? phib : 0.0; break;
    case 2: {
        const double ar = a * r, i1 = ar < 1.0 ? ar : 1.0, t = i1 > 0.0 ? i1 : 0.0, u = r < a ? r : a;
        const bool up = u > t, isq = !up && i1 > 0.0 && ar < 1.0;
        o.r = up && r < a ? phib : isq ? phib * a : 0.0;
        o.a = up && !(r < a) ? phib : isq ? phib * r : 0.0;
        break;
    }
    case 3: {
        const double sg = r < 0.0 ? -1.0 : 1.0, den = 1.0 + fabs(r), c = (r + fabs(r)) / den;
        low3(c, ((1.0 + sg) - c * sg) / den, 0.0, 0.0);
        break;
    }
    case 4: low3((1.0 + r) / 2.0, 0.5, 0.0, 0.0); break;
    case 5: {
        const double den = 1.0 + r * r, c = (r * r + r) / den;
        high2(c, ((2.0 * r + 1.0) - c * 2.0 * r) / den, 0.0);
        break;
    }
    case 6: high2(a < 1.5 ? a : 1.5, 0.0, a < 1.5 ? 1.0 : 0.0); break;
    case 7: low3((1.0 + 2.0 * r) / 3.0, 2.0 / 3.0, 0.0, 0.0); break;
    case 8: low3(ic5, 24.0 / 30.0, -2.0 / 30.0, -3.0 / 30.0); break;
    case 9: o.r = phib * (2.0 / 3.0); break;
    case 10: o.r = phib * (24.0 / 30.0); o.r1 = -(phib * (2.0 / 30.0)); o.r2 = -(phib * (3.0 / 30.0)); break;
    default: break;
    }
    return o;
}

// Bars of one variable's reconstruction: of the fourteen stencil points
// muscl_var reads by themselves, and of the one extremum point each side's
// MLP bound can select (ll of the first point that attains it; 0: none).
struct ReconBar {
    double x9, x10, x23, x32, x37, x38;              // the six along the normal
    double x3, x4, x7, x8, x11, x12, x15, x16;       // the transverse ratios (MLP)
    double el, er;                                   // the bars of the extrema ll = il, ir
    int il, ir;
};

// muscl_var backwards: wl, wr the bars of the left and right values
template <bool MLP, class F> HD ReconBar muscl_back(int nlim, F xs, double wl, double wr)
{
    const double eps = 1.0e-30;
    const double x9 = xs(9), x10 = xs(10), x23 = xs(23), x32 = xs(32);
    const double dq = x10 - x9, dqm = x9 - x23, dqm1 = x23 - xs(37), dqp = x32 - x10, dqp1 = xs(38) - x32;
    LimState<double> m;
    const double im = 1.0 / (dqm + eps), ip = 1.0 / (dqp + eps);
    m.r[0] = dq * im; m.r1[0] = dqm1 * im; m.r2[0] = dqp * im;
    m.r[1] = dq * ip; m.r1[1] = dqp1 * ip; m.r2[1] = dqm * ip;
    m.alp[0] = m.alp[1] = 2.0;
    ReconBar o;
    o.x3 = o.x4 = o.x7 = o.x8 = o.x11 = o.x12 = o.x15 = o.x16 = o.el = o.er = 0.0;
    o.il = o.ir = 0;
    // forward pieces of the MLP bound
    double dyl = 0, dzl = 0, dyr = 0, dzr = 0, nl = 1, nr = 1, A0 = 0, A1 = 0, d1 = 1, d2 = 1, qml = 0, qmr = 0, vl = 0, vr = 0;
    int gl = 0, gr = 0;       // group the selected extremum comes from: 1 ll 1..18, 2 odd of them, 3 even, 4 19..27, 5 28..36
    if constexpr (MLP) {
        const double eps2 = 1.0e-3;
        nl = x10 - x23 + eps;
        nr = x32 - x9 + eps;
        dyl = (xs(11) - xs(7)) / nl;
        dzl = (xs(15) - xs(3)) / nl;
        dyr = (xs(12) - xs(8)) / nr;
        dzr = (xs(16) - xs(4)) / nr;
        const double ryl = fabs(dyl), rzl = fabs(dzl), ryr = fabs(dyr), rzr = fabs(dzr);
        const MlpExt<double> e = mlp_extrema<double>(xs);
        const double a18 = e.a18, b18 = e.b18, aL = e.aL, bL = e.bL, aR = e.aR, bR = e.bR, ao = e.ao, bo = e.bo, ae = e.ae, be = e.be;
        double lo, hi;
        int glo, ghi;
        auto lower = [&](double p, int gp, double q, int gq) { lo = mn(p, q); glo = q < p ? gq : gp; };
        auto upper = [&](double p, int gp, double q, int gq) { hi = mx(p, q); ghi = q > p ? gq : gp; };
        if (ryl < eps2 && rzl < eps2) { lower(a18, 1, aL, 4); upper(b18, 1, bL, 4); }
        else if ((x10 - x23) > 0.0) { hi = b18; ghi = 1; lower(ao, 2, aL, 4); }
        else { lo = a18; glo = 1; upper(bo, 2, bL, 4); }
        {
            const double u = fabs(hi - x9), w = fabs(lo - x9);
            const bool low = w < u;
            qml = low ? w : u;
            vl = low ? lo : hi;
            gl = low ? glo : ghi;
        }
        if (ryr < eps2 && rzr < eps2) { lower(a18, 1, aR, 5); upper(b18, 1, bR, 5); }
        else if ((x32 - x9) > 0.0) { upper(be, 3, bR, 5); lo = a18; glo = 1; }
        else { lower(ae, 3, aR, 5); hi = b18; ghi = 1; }
        {
            const double u = fabs(hi - x10), w = fabs(lo - x10);
            const bool low = w < u;
            qmr = low ? w : u;
            vr = low ? lo : hi;
            gr = low ? glo : ghi;
        }
        d1 = 1.0 + ryl + rzl;
        d2 = 1.0 + ryr + rzr;
        A0 = 2.0 * mx(1.0, m.r[0]) / (fabs(dq) + eps) / d1 * qml;
        if (fabs(dq) <= eps) A1 = 2.0 * mx(1.0, dqp / eps) * fabs(ip) / d2 * qmr;
        else A1 = 2.0 * mx(1.0, 1.0 / m.r[1]) * fabs(ip) / d2 * qmr;
        m.alp[0] = mx(1.0, mn(2.0, A0));
        m.alp[1] = mx(1.0, mn(2.0, A1));
    }
    // backwards
    const double phi0 = limiter(nlim, m, 0), phi1 = limiter(nlim, m, 1);
    double b9 = wl, b10 = wr, dqb = 0.0, dqmb = 0.5 * phi0 * wl, dqpb = -(0.5 * phi1 * wr), imb, ipb;
    const LimBar lb = limiter_back(nlim, m, 0, 0.5 * dqm * wl), rb = limiter_back(nlim, m, 1, -(0.5 * dqp * wr));
    double r0 = lb.r, rR = rb.r, ipx = 0;
    const double r10 = lb.r1, r20 = lb.r2, a0 = lb.a, r1R = rb.r1, r2R = rb.r2, aR = rb.a;
    if constexpr (MLP) {
        double b23 = 0.0, b32 = 0.0;
        // the first point of group gq that holds value v: one bit a point
        // (lo: ll 1..18, hi: the nine of the side's plane), then the group's mask
        auto first = [&](int gq, double v, int plane) {
            unsigned lo = 0, hi = 0;
#pragma unroll
            for (int q = 0; q < 18; q++) lo |= xs(q + 1) == v ? 1u << q : 0u;
#pragma unroll
            for (int q = 0; q < 9; q++) hi |= xs(plane + q) == v ? 1u << q : 0u;
            lo &= gq == 1 ? 0x3FFFFu : gq == 2 ? 0x15555u : gq == 3 ? 0x2AAAAu : 0u;
            hi = gq >= 4 ? hi : 0u;
            return lo ? __builtin_ctz(lo) + 1 : hi ? __builtin_ctz(hi) + plane : 0;
        };
        if (a0 != 0.0 && A0 < 2.0 && A0 > 1.0) {
            const double ab = a0 * A0;
            if (m.r[0] > 1.0) r0 += ab / m.r[0];
            dqb -= ab * (dq < 0.0 ? -1.0 : 1.0) / (fabs(dq) + eps);
            const double db = -(ab / d1);
            const double yb = (dyl < 0.0 ? -db : db) / nl, zb = (dzl < 0.0 ? -db : db) / nl;
            o.x11 += yb; o.x7 -= yb; o.x15 += zb; o.x3 -= zb;
            const double nb = -(yb * dyl + zb * dzl);
            b10 += nb; b23 -= nb;
            const double qb = (vl - x9 < 0.0 ? -1.0 : 1.0) * (ab / qml);
            o.el = qb; o.il = first(gl, vl, 19);
            b9 -= qb;
        }
        if (aR != 0.0 && A1 < 2.0 && A1 > 1.0) {
            const double ab = aR * A1;
            if (fabs(dq) <= eps) {
                if (dqp / eps > 1.0) dqpb += ab / dqp;
            } else if (1.0 / m.r[1] > 1.0) rR -= ab / m.r[1];
            ipx = ab / ip;
            const double db = -(ab / d2);
            const double yb = (dyr < 0.0 ? -db : db) / nr, zb = (dzr < 0.0 ? -db : db) / nr;
            o.x12 += yb; o.x8 -= yb; o.x16 += zb; o.x4 -= zb;
            const double nb = -(yb * dyr + zb * dzr);
            b32 += nb; b9 -= nb;
            const double qb = (vr - x10 < 0.0 ? -1.0 : 1.0) * (ab / qmr);
            o.er = qb; o.ir = first(gr, vr, 28);
            b10 -= qb;
        }
        o.x23 = b23; o.x32 = b32;
    } else {
        o.x23 = o.x32 = 0.0;
    }
    imb = r0 * dq + r10 * dqm1 + r20 * dqp;
    ipb = ipx + rR * dq + r1R * dqp1 + r2R * dqm;
    dqb += r0 * im + rR * ip;
    dqpb += r20 * im - ipb * (ip * ip);
    dqmb += r2R * ip - imb * (im * im);
    const double dqm1b = r10 * im, dqp1b = r1R * ip;
    o.x9 = b9 - dqb + dqmb;
    o.x10 = b10 + dqb - dqpb;
    o.x23 += dqm1b - dqmb;
    o.x32 += dqpb - dqp1b;
    o.x37 = -dqm1b;
    o.x38 = dqp1b;
    return o;
}

// ------------------------------------------------------------ fluxes
// slopes of sndp2(P, snd2, u2) with respect to snd2, u2 and u_ref
struct Sndp2x { double c, u, r; };
HD Sndp2x sndp2_slopes(const Par &P, double snd2, double u2)
{
    if (P.prec == 0) return {1.0, 0.0, 0.0};
    const double ur2 = P.uref * P.uref;
    bool fixed = false;
    double m = ur2 > u2 ? ur2 : u2;
    if (P.prec != 1 && P.str * P.str > m) { m = P.str * P.str; fixed = true; }
    if (!(m < snd2)) return {1.0, 0.0, 0.0};
    if (fixed) return {0.0, 0.0, 0.0};
    if (ur2 > u2) return {0.0, 0.0, 2.0 * P.uref};
    return {0.0, 1.0, 0.0};
}

// bars of a flux core's inputs
struct FluxBar {
    double pl[NPV], pr[NPV], rl, hl, rr, hr, c2, uref;
};

// The mean sound speed squared is the one input whose slopes are formed
// forwards, before the bars are known: at low Mach number they are small
// differences of large terms, and d c^2 / d y1 (some 1e11 in a bubbly mixture)
// multiplies their rounding, which so is the same for every bar (the product
// stays linear in res_bar to rounding of the result, not of those terms).

// ausm_flux backwards; g: the bars of the flux
HD void ausm_back(const Par &P, int npv, const double *n3, const FaceState<double> &L, const FaceState<double> &Rt, double c2avg,
                  const double *g, FluxBar &o)
{
    for (int k = 0; k < NPV; k++) o.pl[k] = o.pr[k] = 0.0;
    o.rl = o.hl = o.rr = o.hr = o.c2 = o.uref = 0.0;
    const double beta = 0.125, kp = 0.25;
    const double dl = sqrt(n3[0] * n3[0] + n3[1] * n3[1] + n3[2] * n3[2]);
    if (dl == 0.0) return;
    const double nx = n3[0] / dl, ny = n3[1] / dl, nz = n3[2] / dl;
    const double *pl = L.p, *pr = Rt.p;
    const double uull = nx * pl[1] + ny * pl[2] + nz * pl[3], uurr = nx * pr[1] + ny * pr[2] + nz * pr[3];
    const double sl = sqrt(L.rho), sr = sqrt(Rt.rho), ravd = 1.0 / (sl + sr);
    const double ua = (sl * pl[1] + sr * pr[1]) * ravd, va = (sl * pl[2] + sr * pr[2]) * ravd, wa = (sl * pl[3] + sr * pr[3]) * ravd;
    const double rr = sqrt(L.rho * Rt.rho), amid = sqrt(c2avg);
    const double zmr = uurr / amid, zml = uull / amid;
    const double un = nx * ua + ny * va + nz * wa, am2 = un * un;
    const double am2r = sndp2(P, c2avg, am2) / c2avg, sq = sqrt(am2r), fmid = sq * (2.0 - sq);
    const double al0 = 0.1875 * (-4.0 + 5.0 * (fmid * fmid));
    const double alpha = mx(mn(al0, 0.1875), -0.75);
    const bool al_on = !(0.1875 < al0) && !(-0.75 > al0);
    double zmmr, pmr, zmmr_z, pmr_z, pmr_a, zmpl, ppl, zmpl_z, ppl_z, ppl_a;
    if (fabs(zmr) >= 1.0) {
        const double s = zmr < 0.0 ? -1.0 : 1.0;
        zmmr = 0.5 * (zmr - fabs(zmr)); pmr = 0.5 * (1.0 - zmr / fabs(zmr));
        zmmr_z = 0.5 * (1.0 - s); pmr_z = 0.0; pmr_a = 0.0;
    } else {
        const double z1 = zmr - 1.0, t1 = z1 * z1, w = zmr * zmr - 1.0, t2 = w * w, t2z = 4.0 * zmr * w;
        zmmr = -(0.25 * t1) - beta * t2; pmr = 0.25 * t1 * (2.0 + zmr) - alpha * zmr * t2;
        zmmr_z = -(0.5 * z1) - beta * t2z;
        pmr_z = 0.25 * (2.0 * z1 * (2.0 + zmr) + t1) - alpha * (t2 + zmr * t2z);
        pmr_a = -(zmr * t2);
    }
    if (fabs(zml) >= 1.0) {
        const double s = zml < 0.0 ? -1.0 : 1.0;
        zmpl = 0.5 * (zml + fabs(zml)); ppl = 0.5 * (1.0 + zml / fabs(zml));
        zmpl_z = 0.5 * (1.0 + s); ppl_z = 0.0; ppl_a = 0.0;
    } else {
        const double z1 = zml + 1.0, t1 = z1 * z1, w = zml * zml - 1.0, t2 = w * w, t2z = 4.0 * zml * w;
        zmpl = 0.25 * t1 + beta * t2; ppl = 0.25 * t1 * (2.0 - zml) + alpha * zml * t2;
        zmpl_z = 0.5 * z1 + beta * t2z;
        ppl_z = 0.25 * (2.0 * z1 * (2.0 - zml) - t1) + alpha * (t2 + zml * t2z);
        ppl_a = zml * t2;
    }
    const double e = 1.0 - am2 / c2avg, f1 = mx(e, 0.0), dP = pr[0] - pl[0], du = uurr - uull;
    const double it = 1.0 / (rr * c2avg * fmid), T = kp * f1 * dP * it;
    const double zmid = zmpl + zmmr - T;
    const bool left = zmid > 0.0;
    const double ml = left ? zmid * amid * L.rho : 0.0, mr = left ? 0.0 : zmid * amid * Rt.rho;
    const double hl = L.h + 0.5 * (pl[1] * pl[1] + pl[2] * pl[2] + pl[3] * pl[3]);
    const double hr = Rt.h + 0.5 * (pr[1] * pr[1] + pr[2] * pr[2] + pr[3] * pr[3]);
    // the flux
    double mlb = (g[0] + g[1] * pl[1] + g[2] * pl[2] + g[3] * pl[3] + g[4] * hl) * dl;
    double mrb = (g[0] + g[1] * pr[1] + g[2] * pr[2] + g[3] * pr[3] + g[4] * hr) * dl;
    const double hlb = ml * g[4] * dl, hrb = mr * g[4] * dl, pmb = (g[1] * nx + g[2] * ny + g[3] * nz) * dl;
    for (int k = 1; k <= 3; k++) {
        o.pl[k] = ml * g[k] * dl + hlb * pl[k];
        o.pr[k] = mr * g[k] * dl + hrb * pr[k];
    }
#pragma unroll
    for (int k = 5; k < NPV; k++) if (k < npv) {
        mlb += g[k] * pl[k] * dl;
        mrb += g[k] * pr[k] * dl;
        o.pl[k] = ml * g[k] * dl;
        o.pr[k] = mr * g[k] * dl;
    }
    o.hl = hlb; o.hr = hrb;
    double zb;
    if (left) { zb = mlb * amid * L.rho; o.rl += mlb * zmid * amid; }
    else { zb = mrb * amid * Rt.rho; o.rr += mrb * zmid * amid; }
    const Sndp2x sx = sndp2_slopes(P, c2avg, am2);
    {   // d / d c2avg, forwards
        const double am_c = 0.5 / amid, zmr_c = -(zmr / amid * am_c), zml_c = -(zml / amid * am_c);
        const double fm_c = sq > 0.0 ? (2.0 - 2.0 * sq) * (0.5 / sq) * ((sx.c - am2r) / c2avg) : 0.0;
        const double al_c = al_on ? 1.875 * fmid * fm_c : 0.0;
        const double pmr_c = pmr_z * zmr_c + pmr_a * al_c, ppl_c = ppl_z * zml_c + ppl_a * al_c;
        const double f1_c = !(0.0 > e) ? am2 / (c2avg * c2avg) : 0.0;
        const double T_c = kp * f1_c * dP * it - T / c2avg - T / fmid * fm_c;
        const double zm_c = zmpl_z * zml_c + zmmr_z * zmr_c - T_c, m_c = zm_c * amid + zmid * am_c;
        const double pm_c = ppl_c * (pl[0] + P.pref) + pmr_c * (pr[0] + P.pref)
                          - 2.0 * rr * du * ((ppl_c * pmr + ppl * pmr_c) * fmid * amid + ppl * pmr * (fm_c * amid + fmid * am_c));
        o.c2 = (left ? mlb * L.rho : mrb * Rt.rho) * m_c + pmb * pm_c;
    }
    // pmid
    const double X = 2.0 * ppl * pmr;
    const double pplb = pmb * (pl[0] + P.pref - 2.0 * pmr * rr * fmid * amid * du);
    const double pmrb = pmb * (pr[0] + P.pref - 2.0 * ppl * rr * fmid * amid * du);
    o.pl[0] += pmb * ppl;
    o.pr[0] += pmb * pmr;
    double rrb = -(pmb * X * fmid * amid * du), fb = -(pmb * X * rr * amid * du);
    const double dub = -(pmb * X * rr * fmid * amid);
    // zmid's pressure diffusion
    const double Tb = -zb, dPb = Tb * kp * f1 * it;
    rrb -= Tb * T / rr;
    fb -= Tb * T / fmid;
    o.pr[0] += dPb;
    o.pl[0] -= dPb;
    double am2b = 0.0;
    if (!(0.0 > e)) am2b -= Tb * kp * dP * it / c2avg;
    // the split Mach numbers and pressures
    const double zmrb = zb * zmmr_z + pmrb * pmr_z, zmlb = zb * zmpl_z + pplb * ppl_z;
    if (al_on) fb += (pmrb * pmr_a + pplb * ppl_a) * 1.875 * fmid;
    const double uurrb = dub + zmrb / amid, uullb = zmlb / amid - dub;
    // fmid = sq (2 - sq), sq = sqrt(sndp2 / c2)
    const double spb = sq > 0.0 ? fb * (2.0 - 2.0 * sq) * (0.5 / sq) / c2avg : 0.0;
    am2b += spb * sx.u;
    o.uref = spb * sx.r;
    const double unb = 2.0 * un * am2b, nv[3] = {nx, ny, nz}, av[3] = {ua, va, wa};
    double slb = 0.0, srb = 0.0;
    for (int k = 0; k < 3; k++) {
        const double q = unb * nv[k] * ravd;
        o.pl[k + 1] += q * sl + nv[k] * uullb;
        o.pr[k + 1] += q * sr + nv[k] * uurrb;
        slb += q * (pl[k + 1] - av[k]);
        srb += q * (pr[k + 1] - av[k]);
    }
    o.rl += rrb * 0.5 * Rt.rho / rr + slb * (0.5 / sl);
    o.rr += rrb * 0.5 * L.rho / rr + srb * (0.5 / sr);
}

// roe_flux backwards
HD void roe_back(const Par &P, int npv, const double *n3, const FaceState<double> &L, const FaceState<double> &Rt, double c2avg,
                 const double *g, FluxBar &o)
{
    for (int k = 0; k < NPV; k++) o.pl[k] = o.pr[k] = 0.0;
    o.rl = o.hl = o.rr = o.hr = o.c2 = o.uref = 0.0;
    const double dl = sqrt(n3[0] * n3[0] + n3[1] * n3[1] + n3[2] * n3[2]);
    if (dl == 0.0) return;
    const double nv[3] = {n3[0] / dl, n3[1] / dl, n3[2] / dl};
    const double *pl = L.p, *pr = Rt.p;
    const double uull = nv[0] * pl[1] + nv[1] * pl[2] + nv[2] * pl[3], uurr = nv[0] * pr[1] + nv[1] * pr[2] + nv[2] * pr[3];
    const double sl = sqrt(L.rho), sr = sqrt(Rt.rho), ravd = 1.0 / (sl + sr);
    double ra[NPV], rab[NPV];
    for (int k = 0; k < NPV; k++) ra[k] = rab[k] = 0.0;
#pragma unroll
    for (int k = 1; k < NPV; k++) if (k != 4 && k < npv) ra[k] = (sl * pl[k] + sr * pr[k]) * ravd;
    const double hl = L.h + 0.5 * (pl[1] * pl[1] + pl[2] * pl[2] + pl[3] * pl[3]);
    const double hr = Rt.h + 0.5 * (pr[1] * pr[1] + pr[2] * pr[2] + pr[3] * pr[3]);
    const double raht = (sl * hl + sr * hr) * ravd;
    const double u2 = ra[1] * ra[1] + ra[2] * ra[2] + ra[3] * ra[3];
    const double rr = sqrt(L.rho * Rt.rho);
    const double uuu = nv[0] * ra[1] + nv[1] * ra[2] + nv[2] * ra[3];
    const double sp = sndp2(P, c2avg, u2), q = sp / c2avg, omq = 1.0 - q, uup = 0.5 * (1.0 + q) * uuu;
    const double rt = sqrt(omq * omq * (uuu * uuu) + 4.0 * sp), ddd = 0.5 * rt;
    const double A = uup + ddd, Bm = uup - ddd, sA = A < 0.0 ? -1.0 : 1.0, sB = Bm < 0.0 ? -1.0 : 1.0;
    const double cs = 0.5 * (fabs(A) + fabs(Bm)), ms = 0.5 * (fabs(A) - fabs(Bm)) / ddd;
    const double dpp = pr[0] - pl[0], dun = uurr - uull, au = fabs(uuu), s = uuu < 0.0 ? -1.0 : 1.0;
    const double C1 = cs - q * au - 0.5 * omq * uuu * ms, C2 = cs - au + 0.5 * omq * uuu * ms;
    const double isp = 1.0 / (rr * sp), K = dpp * isp;
    const double du = ms * dun + C1 * K, dp = ms * dpp + C2 * rr * dun, dur = du * rr;
    const double ml = L.rho * uull, mr = Rt.rho * uurr, hg = 0.5 * dl;
    // the flux: ml ql + mr qr - au (rhoR qr - rhoL ql) - dur qa for every equation
    double mlb = 0.0, mrb = 0.0, aub = 0.0, durb = 0.0, uuub = 0.0, rahtb, hlb, hrb;
    auto eq = [&](double gs, double ql, double qr, double qa, double &qlb, double &qrb, double &qab) {
        mlb += gs * ql; mrb += gs * qr;
        qlb += gs * (ml + au * L.rho); qrb += gs * (mr - au * Rt.rho); qab -= gs * dur;
        aub -= gs * (Rt.rho * qr - L.rho * ql);
        durb -= gs * qa;
        o.rr -= gs * au * qr; o.rl += gs * au * ql;
    };
    double x0 = 0, x1 = 0, x2 = 0;
    eq(hg * g[0], 1.0, 1.0, 1.0, x0, x1, x2);
#pragma unroll
    for (int k = 1; k < NPV; k++) if (k != 4 && k < npv) eq(hg * g[k], pl[k], pr[k], ra[k], o.pl[k], o.pr[k], rab[k]);
    hlb = hrb = rahtb = 0.0;
    eq(hg * g[4], hl, hr, raht, hlb, hrb, rahtb);
    const double g4 = hg * g[4], gn = hg * (g[1] * nv[0] + g[2] * nv[1] + g[3] * nv[2]);
    o.pr[0] += g4 * au + gn;
    o.pl[0] += gn - g4 * au;
    aub -= g4 * (pl[0] - pr[0]);
    const double dpb = -(gn + g4 * uuu);
    uuub -= g4 * dp;
    // dur, du, dp
    const double dub = durb * rr;
    double rrb = durb * du;
    uuub += aub * s;
    const double C2b = dpb * rr * dun, C1b = dub * K, Kb = dub * C1;
    double msb = dpb * dpp + dub * dun, csb = C1b + C2b, dppb = dpb * ms + Kb * isp, dunb = dpb * C2 * rr + dub * ms;
    rrb += dpb * C2 * dun - Kb * K / rr;
    double spb = -(Kb * K / sp), qb = -(C1b * au);
    uuub -= C2b * s + C1b * q * s;
    const double hb = 0.5 * (C2b - C1b);
    double omqb = hb * uuu * ms;
    uuub += hb * omq * ms;
    msb += hb * omq * uuu;
    // cs, ms
    const double mh = msb * 0.5 / ddd, tA = sA * (0.5 * csb + mh), tB = sB * (0.5 * csb - mh);
    double dddb = -(msb * ms / ddd) + tA - tB;
    const double uupb = tA + tB;
    const double Eb = dddb * 0.25 / rt;
    omqb += Eb * 2.0 * omq * (uuu * uuu);
    uuub += Eb * 2.0 * (omq * omq) * uuu;
    spb += 4.0 * Eb;
    qb += uupb * 0.5 * uuu - omqb;
    uuub += uupb * 0.5 * (1.0 + q);
    spb += qb / c2avg;
    const Sndp2x sx = sndp2_slopes(P, c2avg, u2);
    const double u2b = spb * sx.u;
    o.uref = spb * sx.r;
    {   // d / d c2avg, forwards
        const double q_c = (sx.c - q) / c2avg, up_c = 0.5 * q_c * uuu;
        const double dd_c = 0.25 / rt * (4.0 * sx.c - 2.0 * omq * q_c * (uuu * uuu));
        const double A_c = sA * (up_c + dd_c), B_c = sB * (up_c - dd_c);
        const double cs_c = 0.5 * (A_c + B_c), ms_c = (0.5 * (A_c - B_c) - ms * dd_c) / ddd, h_c = 0.5 * uuu * (omq * ms_c - q_c * ms);
        o.c2 = dub * (ms_c * dun + (cs_c - q_c * au - h_c) * K - C1 * K * sx.c / sp) + dpb * (ms_c * dpp + (cs_c + h_c) * rr * dun);
    }
    double slb = rahtb * (hl - raht) * ravd, srb = rahtb * (hr - raht) * ravd;
    hlb += rahtb * sl * ravd;
    hrb += rahtb * sr * ravd;
    o.pr[0] += dppb;
    o.pl[0] -= dppb;
    const double uurrb = dunb + mrb * Rt.rho, uullb = mlb * L.rho - dunb;
    o.rl += mlb * uull;
    o.rr += mrb * uurr;
    for (int k = 1; k <= 3; k++) {
        rab[k] += 2.0 * ra[k] * u2b + nv[k - 1] * uuub;
        o.pl[k] += nv[k - 1] * uullb + hlb * pl[k];
        o.pr[k] += nv[k - 1] * uurrb + hrb * pr[k];
    }
#pragma unroll
    for (int k = 1; k < NPV; k++) if (k != 4 && k < npv) {
        const double w = rab[k] * ravd;
        o.pl[k] += w * sl;
        o.pr[k] += w * sr;
        slb += w * (pl[k] - ra[k]);
        srb += w * (pr[k] - ra[k]);
    }
    o.hl = hlb; o.hr = hrb;
    o.rl += rrb * 0.5 * Rt.rho / rr + slb * (0.5 / sl);
    o.rr += rrb * 0.5 * L.rho / rr + srb * (0.5 / sr);
}

// roem_flux / ausmpwp_flux: two-lane dual passes over {pL, pR, rhoL, hL, rhoR,
// hR, c2avg, c2L, c2R, sd[18], u_ref}
HD void sensor_back(const Par &P, int npv, const double *n3, const FaceState<double> &L, const FaceState<double> &Rt, double c2avg,
                    const double *sd, const double *g, FluxBar &b, double &c2lb, double &c2rb, double *sdb)
{
    constexpr int NZ = 2 * NPV + 26, W = 2;
    using T = Dn<W>;
    const int o = 2 * npv, nz = o + 26;
    double zx[NZ], zb[NZ];
    for (int n = 0; n < npv; n++) { zx[n] = L.p[n]; zx[npv + n] = Rt.p[n]; }
    zx[o] = L.rho; zx[o + 1] = L.h; zx[o + 2] = Rt.rho; zx[o + 3] = Rt.h; zx[o + 4] = c2avg;
    zx[o + 5] = L.c2; zx[o + 6] = Rt.c2;
    for (int q = 0; q < 18; q++) zx[o + 7 + q] = sd[q];
    zx[nz - 1] = P.uref;
    dn_grad<W>(nz, [&](int q) -> double { return zx[q]; }, [&](auto in, int base) -> T {
        FaceState<T> l, r;
        for (int n = 0; n < NPV; n++) {
            l.p[n] = n < npv ? in(n) : T(0.0);
            r.p[n] = n < npv ? in(npv + n) : T(0.0);
        }
        l.rho = in(o); l.h = in(o + 1); r.rho = in(o + 2); r.h = in(o + 3);
        l.c2 = in(o + 5);
        r.c2 = in(o + 6);
        Par Pu = P;
        const int lu = nz - 1 - base;
        Pu.uref_seed = (lu >= 0 && lu < W) ? lu + 1 : 0;
        const T nt[3] = {T(n3[0]), T(n3[1]), T(n3[2])};
        T fx[NPV], sdt[18];
        for (int q = 0; q < 18; q++) sdt[q] = in(o + 7 + q);
        if (P.nscheme == 2) roem_flux<T>(Pu, npv, nt, l, r, in(o + 4), sdt, fx);
        else ausmpwp_flux<T>(Pu, npv, nt, l, r, in(o + 4), sdt, fx);
        T phi(0.0);
        for (int n = 0; n < npv; n++) phi = phi + g[n] * fx[n];
        return phi;
    }, zb);
    for (int n = 0; n < NPV; n++) { b.pl[n] = n < npv ? zb[n] : 0.0; b.pr[n] = n < npv ? zb[npv + n] : 0.0; }
    b.rl = zb[o]; b.hl = zb[o + 1]; b.rr = zb[o + 2]; b.hr = zb[o + 3]; b.c2 = zb[o + 4];
    c2lb = zb[o + 5]; c2rb = zb[o + 6];
    for (int q = 0; q < 18; q++) sdb[q] = zb[o + 7 + q];
    b.uref = zb[nz - 1];
}

// Bars a face leaves behind: of its reconstructed (or, where a clamp or a
// first-order face took them, the cells') left and right values, of the
// sensor pressures, of the cells' rho, h, c^2 (first-order faces) and of u_ref.
struct FaceBar {
    double wl[NPV], wr[NPV];
    int cell;                 // bit n: wl[n] belongs to the left cell's own value; bit 16 + n: wr[n] to the right's
    double sen[18];
    double prop[2][3];        // rho, h, c^2 of the left and right cells
    double uref;
};

// The inviscid adjoint of one face up to its reconstruction, independent of
// its direction: xs(ll, n) the stencil values; cellp = {rho, h, c^2} of the
// left and right cells (read by first-order faces); g the seed of the flux.
template <bool SENSOR, class X>
__host__ __device__ __attribute__((always_inline)) inline void face_adj_core(const Par &P, int npv, X xs, const double *n3,
                                      const double *cellp, const double *g, FaceBar &o)
{
    // forward recompute: reconstruction, clamps, face EOS, averaged c^2
    FaceState<double> L, Rt;
    int ol[NPV], orr[NPV];
    double dl[ND], dr[ND];
    {
        double c9[NPV], c10[NPV], g3[6][3];
        Par Pi = P;
        Pi.iturb = -3;
        for (int n = 0; n < NPV; n++) { L.p[n] = Rt.p[n] = 0.0; ol[n] = orr[n] = 1; c9[n] = c10[n] = 0.0; }
        face_recon<double>(Pi, npv, xs, c9, c10, L.p, Rt.p, g3);
        if (P.nmuscl > 0) clamps_src(npv, P.pref, c9, c10, L.p, Rt.p, ol, orr);
    }
    if (P.nmuscl > 0) {
        // rho and h of the face states with the mixture's own derivatives
        // (d rho/dp, ...; dh/dp, ...), their exact gradients
        mixture_eos<double>(L.p[0] + P.pref, L.p[4], L.p[5], L.p[6], dl, false);
        mixture_eos<double>(Rt.p[0] + P.pref, Rt.p[4], Rt.p[5], Rt.p[6], dr, false);
        L.rho = dl[D_RHO]; L.h = dl[D_H]; L.c2 = dl[D_C2];
        Rt.rho = dr[D_RHO]; Rt.h = dr[D_H]; Rt.c2 = dr[D_C2];
    } else {
        L.rho = cellp[0]; L.h = cellp[1]; L.c2 = cellp[2];
        Rt.rho = cellp[3]; Rt.h = cellp[4]; Rt.c2 = cellp[5];
    }
    const double sl = sqrt(L.rho), sr = sqrt(Rt.rho), rd = 1.0 / (sl + sr);
    const double pa = 0.5 * (L.p[0] + Rt.p[0]) + P.pref, ta = 0.5 * (L.p[4] + Rt.p[4]);
    const double ya1 = (sl * L.p[5] + sr * Rt.p[5]) * rd, ya2 = (sl * L.p[6] + sr * Rt.p[6]) * rd;
    const double c2a = face_c2<double>(pa, ta, ya1, ya2);
    FluxBar b;
    double c2lb = 0.0, c2rb = 0.0;
    if constexpr (SENSOR) {
        double sd[18];
        for (int ll = 1; ll <= 18; ll++) sd[ll - 1] = xs(ll, 0);
        sensor_back(P, npv, n3, L, Rt, c2a, sd, g, b, c2lb, c2rb, o.sen);
    } else {
        if (P.nscheme == 1) roe_back(P, npv, n3, L, Rt, c2a, g, b);
        else ausm_back(P, npv, n3, L, Rt, c2a, g, b);
    }
    o.uref = b.uref;
    {   // averaged c^2 back to the averaged state, then the Roe averages
        double g4[4];
        c2_back(pa, ta, ya1, ya2, b.c2, g4);
        b.pl[0] += 0.5 * g4[0]; b.pr[0] += 0.5 * g4[0];
        b.pl[4] += 0.5 * g4[1]; b.pr[4] += 0.5 * g4[1];
        b.pl[5] += g4[2] * sl * rd; b.pr[5] += g4[2] * sr * rd;
        b.pl[6] += g4[3] * sl * rd; b.pr[6] += g4[3] * sr * rd;
        // d ya / d sl = (x_L - ya) / (sl + sr), d sl / d rho_L = 0.5 / sl
        b.rl += (g4[2] * (L.p[5] - ya1) + g4[3] * (L.p[6] - ya2)) * rd * (0.5 / sl);
        b.rr += (g4[2] * (Rt.p[5] - ya1) + g4[3] * (Rt.p[6] - ya2)) * rd * (0.5 / sr);
    }
    for (int q = 0; q < 3; q++) o.prop[0][q] = o.prop[1][q] = 0.0;
    if (P.nmuscl > 0) {   // face EOS of each side
        b.pl[0] += b.rl * dl[D_RP] + b.hl * dl[D_HP];
        b.pl[4] += b.rl * dl[D_RT] + b.hl * dl[D_HT];
        b.pl[5] += b.rl * dl[D_RY1] + b.hl * dl[D_HY1];
        b.pl[6] += b.rl * dl[D_RY2] + b.hl * dl[D_HY2];
        b.pr[0] += b.rr * dr[D_RP] + b.hr * dr[D_HP];
        b.pr[4] += b.rr * dr[D_RT] + b.hr * dr[D_HT];
        b.pr[5] += b.rr * dr[D_RY1] + b.hr * dr[D_HY1];
        b.pr[6] += b.rr * dr[D_RY2] + b.hr * dr[D_HY2];
        if constexpr (SENSOR) {     // c^2 of the face states
            double gx[4];
            if (c2lb != 0.0) {
                c2_back(L.p[0] + P.pref, L.p[4], L.p[5], L.p[6], c2lb, gx);
                b.pl[0] += gx[0]; b.pl[4] += gx[1]; b.pl[5] += gx[2]; b.pl[6] += gx[3];
            }
            if (c2rb != 0.0) {
                c2_back(Rt.p[0] + P.pref, Rt.p[4], Rt.p[5], Rt.p[6], c2rb, gx);
                b.pr[0] += gx[0]; b.pr[4] += gx[1]; b.pr[5] += gx[2]; b.pr[6] += gx[3];
            }
        }
    } else {
        o.prop[0][0] = b.rl; o.prop[0][1] = b.hl; o.prop[0][2] = c2lb;
        o.prop[1][0] = b.rr; o.prop[1][1] = b.hr; o.prop[1][2] = c2rb;
    }
    // through the clamps to the raw reconstruction or the cells
    o.cell = 0;
    for (int n = 0; n < NPV; n++) {
        o.wl[n] = ol[n] == 2 ? 0.0 : b.pl[n];
        o.wr[n] = orr[n] == 2 ? 0.0 : b.pr[n];
        o.cell |= (ol[n] == 1 ? 1 << n : 0) | (orr[n] == 1 ? 1 << (16 + n) : 0);
    }
}

// The inviscid adjoint of one face on its 38-point stencil (the kernels run
// the two parts separately): f0 points at the left cell's pressure,
// off[ll-1] is stencil point ll's offset and ng the component stride.  Out:
// sbo[(ll-1)*ss + n*sn] the bar of stencil point ll of variable n for every
// ll in mask (bit ll-1), dcbo[(side*ND + m)*dstr] the two cells' property
// bars, ub the u_ref derivative.
template <bool SENSOR>
__host__ __device__ __attribute__((always_inline)) inline void face_adj(const Par &P, int npv, const double *f0, long ng, const long *off, const double *n3,
                                      const double *cellp, const double *g, unsigned long long mask, double *sbo,
                                      long ss, long sn, double *dcbo, long dstr, double &ub)
{
    FaceBar fb;
    face_adj_core<SENSOR>(P, npv, [&](int ll, int n) -> double { return f0[(long)n * ng + off[ll - 1]]; }, n3, cellp, g, fb);
    ub = fb.uref;
    for (int m = 0; m < 2 * ND; m++) dcbo[(long)m * dstr] = 0.0;
    for (int sd = 0; sd < 2; sd++) {
        dcbo[(long)(sd * ND + D_RHO) * dstr] = fb.prop[sd][0];
        dcbo[(long)(sd * ND + D_H) * dstr] = fb.prop[sd][1];
        dcbo[(long)(sd * ND + D_C2) * dstr] = fb.prop[sd][2];
    }
    for (int n = 0; n < npv; n++) {
        double sb[NSLOT];
        for (int q = 0; q < NSLOT; q++) sb[q] = 0.0;
        const bool cl = (fb.cell >> n) & 1, cr = (fb.cell >> (16 + n)) & 1;
        const double wl = cl ? 0.0 : fb.wl[n], wr = cr ? 0.0 : fb.wr[n];
        if (cl) sb[8] += fb.wl[n];
        if (cr) sb[9] += fb.wr[n];
        if (wl != 0.0 || wr != 0.0) {
            auto xs = [&](int ll) -> double { return f0[(long)n * ng + off[ll - 1]]; };
            const ReconBar r = P.nmuscl == 2 ? muscl_back<true>(P.nlim, xs, wl, wr) : muscl_back<false>(P.nlim, xs, wl, wr);
            sb[8] += r.x9; sb[9] += r.x10; sb[22] += r.x23; sb[31] += r.x32; sb[36] += r.x37; sb[37] += r.x38;
            sb[2] += r.x3; sb[3] += r.x4; sb[6] += r.x7; sb[7] += r.x8; sb[10] += r.x11; sb[11] += r.x12; sb[14] += r.x15; sb[15] += r.x16;
            if (r.il) sb[r.il - 1] += r.el;
            if (r.ir) sb[r.ir - 1] += r.er;
        }
        if (SENSOR && n == 0)
            for (int q = 0; q < 18; q++) sb[q] += fb.sen[q];
        for (int ll = 1; ll <= NSLOT; ll++)
            if ((mask >> (ll - 1)) & 1ull) sbo[(long)(ll - 1) * ss + (long)n * sn] = sb[ll - 1];
    }
}

// bars of one face's viscous flux
struct ViscBar {
    double g3[6][3], cav[5];          // normal / transverse differences, face averages
    double mu, kap, ht[2], rho;       // d mu_L = d mu_R = mu, kappa and rho alike (they enter as averages)
    double mut[2];                    // the two cells' eddy viscosities
};

// visc_flux backwards; g: the bars of the flux.  Arguments as visc_flux.
HD void visc_back(const Par &P, const double *nx, const double e4[4][3], const double t4[4][3], const double *gl, const double *gr,
                  const double g3[6][3], const double *cav, const double *dl, const double *dr, double mutl, double mutr,
                  const double *gf, ViscBar &o)
{
    const double c23 = 2.0 / 3.0;
    const bool turb = (P.iturb == 0);
    const int nv = turb ? 6 : 4;
    double em[3], tm[3];
    for (int c = 0; c < 3; c++) {
        em[c] = 0.25 * (e4[0][c] + e4[1][c] + e4[2][c] + e4[3][c]);
        tm[c] = 0.25 * (t4[0][c] + t4[1][c] + t4[2][c] + t4[3][c]);
    }
    const double vol = 2.0 / (gl[0] + gr[0]);
    const double vis = 0.5 * (dl[D_MU] + dr[D_MU]), con = 0.5 * (dl[D_KAP] + dr[D_KAP]);
    const double emut = turb ? 0.5 * (mutl + mutr) : 0.0, tcon = turb ? 0.5 * (mutl * dl[D_HT] + mutr * dr[D_HT]) / 0.9 : 0.0;
    double g[6][3], gb[6][3];
#pragma unroll
    for (int q = 0; q < 6; q++)
        for (int c = 0; c < 3; c++) {
            g[q][c] = q < nv ? (g3[q][0] * nx[c] + g3[q][1] * em[c] + g3[q][2] * tm[c]) * vol : 0.0;
            gb[q][c] = 0.0;
        }
    const double uc = cav[0], vc = cav[1], wc = cav[2], mu = vis + emut, kap = con + tcon;
    const double div = g[0][0] + g[1][1] + g[2][2];
    const double sxx = 2.0 * g[0][0] - c23 * div, syy = 2.0 * g[1][1] - c23 * div, szz = 2.0 * g[2][2] - c23 * div;
    const double sxy = g[0][1] + g[1][0], sxz = g[0][2] + g[2][0], syz = g[1][2] + g[2][1];
    const double a1 = gf[1] + gf[4] * uc, a2 = gf[2] + gf[4] * vc, a3 = gf[3] + gf[4] * wc;
    const double xxb = a1 * nx[0], yyb = a2 * nx[1], zzb = a3 * nx[2];
    const double xyb = a1 * nx[1] + a2 * nx[0], xzb = a1 * nx[2] + a3 * nx[0], yzb = a2 * nx[2] + a3 * nx[1];
    o.cav[0] = gf[4] * mu * (nx[0] * sxx + nx[1] * sxy + nx[2] * sxz);
    o.cav[1] = gf[4] * mu * (nx[0] * sxy + nx[1] * syy + nx[2] * syz);
    o.cav[2] = gf[4] * mu * (nx[0] * sxz + nx[1] * syz + nx[2] * szz);
    o.cav[3] = o.cav[4] = 0.0;
    const double kapb = gf[4] * (nx[0] * g[3][0] + nx[1] * g[3][1] + nx[2] * g[3][2]);
    const double mub = xxb * sxx + yyb * syy + zzb * szz + xyb * sxy + xzb * sxz + yzb * syz;
    const double divb = -(c23 * mu * (xxb + yyb + zzb));
    gb[0][0] = 2.0 * mu * xxb + divb; gb[1][1] = 2.0 * mu * yyb + divb; gb[2][2] = 2.0 * mu * zzb + divb;
    gb[0][1] = gb[1][0] = mu * xyb; gb[0][2] = gb[2][0] = mu * xzb; gb[1][2] = gb[2][1] = mu * yzb;
    for (int c = 0; c < 3; c++) gb[3][c] = gf[4] * kap * nx[c];
    double visb = mub, emutb = turb ? mub : 0.0, rhob = 0.0;
    o.ht[0] = o.ht[1] = o.mut[0] = o.mut[1] = 0.0;
    if (turb) {
        const double pkw = g[4][0] * g[5][0] + g[4][1] * g[5][1] + g[4][2] * g[5][2];
        const double rho = 0.5 * (dl[D_RHO] + dr[D_RHO]), yd = 0.5 * (gl[1] + gr[1]), kk = cav[3], oo = cav[4];
        const double c0 = 1.712 * rho / oo * pkw, cdkw = mx(c0, 1.0e-10), sk = sqrt(kk);
        const double t1 = sk / (0.09 * oo * yd), t2 = 500.0 * vis / rho / (oo * (yd * yd)), t3 = (3.424 * rho * kk) / (cdkw * (yd * yd));
        const double m12 = mx(t1, t2), b1 = mn(m12, t3), b2 = b1 * b1, bf = tanh(b2 * b2);
        const double tdk = bf * 0.85 + (1.0 - bf) * 1.0, tdo = bf * 0.5 + (1.0 - bf) * 0.856;
        const double S7 = g[4][0] * nx[0] + g[4][1] * nx[1] + g[4][2] * nx[2], S8 = g[5][0] * nx[0] + g[5][1] * nx[1] + g[5][2] * nx[2];
        visb += gf[7] * S7 + gf[8] * S8;
        emutb += gf[7] * tdk * S7 + gf[8] * tdo * S8;
        for (int c = 0; c < 3; c++) {
            gb[4][c] = gf[7] * (vis + emut * tdk) * nx[c];
            gb[5][c] = gf[8] * (vis + emut * tdo) * nx[c];
        }
        const double bfb = gf[7] * emut * S7 * (0.85 - 1.0) + gf[8] * emut * S8 * (0.5 - 0.856);
        const double ab = bfb * (1.0 - bf * bf) * 4.0 * b2 * b1;
        double kb = 0.0, ob = 0.0;
        if (t3 < m12) {
            const double q = 3.424 / (cdkw * (yd * yd));
            rhob += ab * q * kk;
            kb += ab * q * rho;
            if (!(1.0e-10 > c0)) {
                const double cb = -(ab * t3 / cdkw), pb = cb * 1.712 * rho / oo;
                rhob += cb * 1.712 / oo * pkw;
                ob -= cb * c0 / oo;
                for (int c = 0; c < 3; c++) {
                    gb[4][c] += pb * g[5][c];
                    gb[5][c] += pb * g[4][c];
                }
            }
        } else if (t2 > t1) {
            visb += ab * 500.0 / rho / (oo * (yd * yd));
            rhob -= ab * t2 / rho;
            ob -= ab * t2 / oo;
        } else {
            kb += sk > 0.0 ? ab * (0.5 / sk) / (0.09 * oo * yd) : 0.0;
            ob -= ab * t1 / oo;
        }
        o.cav[3] = kb;
        o.cav[4] = ob;
        const double tb = kapb * 0.5 / 0.9;
        o.ht[0] = tb * mutl;
        o.ht[1] = tb * mutr;
        o.mut[0] = 0.5 * emutb + tb * dl[D_HT];
        o.mut[1] = 0.5 * emutb + tb * dr[D_HT];
    }
    o.mu = 0.5 * visb;
    o.kap = 0.5 * kapb;
    o.rho = 0.5 * rhob;
#pragma unroll
    for (int q = 0; q < 6; q++) {
        o.g3[q][0] = q < nv ? vol * (gb[q][0] * nx[0] + gb[q][1] * nx[1] + gb[q][2] * nx[2]) : 0.0;
        o.g3[q][1] = q < nv ? vol * (gb[q][0] * em[0] + gb[q][1] * em[1] + gb[q][2] * em[2]) : 0.0;
        o.g3[q][2] = q < nv ? vol * (gb[q][0] * tm[0] + gb[q][1] * tm[1] + gb[q][2] * tm[2]) : 0.0;
    }
}

// bars of one cell's sources
struct SourceBar {
    double pc[NPV];                   // the cell's own state
    double g[5][3];                   // the gradients of u, v, w, k, omega
    double rho, h, mu, mut;           // its properties and eddy viscosity
    double sc[3];                     // the mass-transfer scales u_ref, dp_ref, t_ref
};

// rb . (the cell's sources) backwards: mass transfer, SST, BDF.  MODELS as
// k_combine.  The sources depend on the cell through few numbers - the
// mass transfer through (p, T, y1, y2, rho) and its three scales, SST through
// k, omega, three properties and SstGrad's invariants of the fifteen gradient
// components - so dual passes run over those of each source alone (one
// sum over all thirty inputs ran every source in each of fifteen two-lane
// passes), and the invariants and the BDF term are transposed by hand.
template <bool MODELS>
HD void source_back(const Par &P, const double *pc, const double *d, const double gr[5][3], const double f6[6][3], double vol,
                    double ydn, double mut, const double *rb, SourceBar &o)
{
    for (int n = 0; n < NPV; n++) o.pc[n] = 0.0;
    for (int v = 0; v < 5; v++) for (int c = 0; c < 3; c++) o.g[v][c] = 0.0;
    o.rho = o.h = o.mu = o.mut = o.sc[0] = o.sc[1] = o.sc[2] = 0.0;
    if (P.ncav >= 1) {
        // p, T, y1, y2, rho, u_ref, dp_ref, t_ref
        constexpr int W = 2;
        using T = Dn<W>;
        const double x[5] = {pc[0], pc[4], pc[5], pc[6], d[D_RHO]};
        double zb[8];
        dn_grad<W>(8, [&](int q) -> double { return q < 5 ? x[q] : 0.0; }, [&](auto in, int base) -> T {
            Par Pu = P;
            auto lane_of = [&](int q) { const int l = q - base; return l >= 0 && l < W ? l + 1 : 0; };
            Pu.uref_seed = lane_of(5);
            Pu.dpref_seed = lane_of(6);
            Pu.tref_seed = lane_of(7);
            T p[NPV], dt[ND], rc, rv, ic[4];
            for (int n = 0; n < NPV; n++) p[n] = T(pc[n]);
            p[0] = in(0); p[4] = in(1); p[5] = in(2); p[6] = in(3);
            bool full_eos = false;
            if constexpr (MODELS)
                if (P.ncav >= 2) {      // on the cell's full EOS, as k_combine<true>
                    T dd[ND], full[18];
                    mixture_eos<T>(p[0] + P.pref, p[4], p[5], p[6], dd, false, full);
                    cav_model<T>(Pu, p, full, vol, rc, rv, ic);
                    full_eos = true;
                }
            if (!full_eos) {
                for (int m = 0; m < ND; m++) dt[m] = T(d[m]);
                dt[D_RHO] = in(4);
                merkle<T>(Pu, p, dt, vol, rc, rv, ic);
            }
            return rb[5] * (rv - rc);
        }, zb);
        o.pc[0] = zb[0]; o.pc[4] = zb[1]; o.pc[5] = zb[2]; o.pc[6] = zb[3];
        o.rho = zb[4];
        const bool sc = P.ncav <= 3;
        for (int q = 0; q < 3; q++) o.sc[q] = sc ? zb[5 + q] : 0.0;
    }
    if (P.iturb == 0) {
        // k, omega, rho, mu, mu_t and the invariants div, S^2, k-omega product (and W^2)
        constexpr int W = MODELS ? 3 : 4, NI = MODELS ? 9 : 8;
        using T = Dn<W>;
        const double *gu = gr[0], *gv = gr[1], *gw = gr[2];
        const SstGrad<double> gi = sst_grad<MODELS, double>(gu, gv, gw, gr[3], gr[4]);
        const double x[9] = {pc[7], pc[8], d[D_RHO], d[D_MU], mut, gi.div, gi.s2, gi.pkw, gi.w2};
        double zb[NI];
        dn_grad<W>(NI, [&](int q) -> double { return x[q]; }, [&](auto in, int) -> T {
            T dt[ND], src[2], it[4], oc;
            for (int m = 0; m < ND; m++) dt[m] = T(d[m]);
            dt[D_RHO] = in(2); dt[D_MU] = in(3);
            const SstGrad<T> g{in(5), in(6), in(7), MODELS ? in(8) : T(0.0)};
            sst_source_i<MODELS, T>(P, g, in(0), in(1), f6, vol, ydn, dt, in(4), src, it, oc);
            return rb[7] * src[0] + rb[8] * src[1];
        }, zb);
        o.pc[7] = zb[0]; o.pc[8] = zb[1];
        o.rho += zb[2]; o.mu = zb[3]; o.mut = zb[4];
        const double s2 = 2.0 * zb[6], w2 = MODELS ? 2.0 * zb[NI - 1] : 0.0;
        for (int c = 0; c < 3; c++) {
            o.g[c][c] = zb[5] + 2.0 * s2 * gr[c][c];
            o.g[3][c] = zb[7] * gr[4][c];
            o.g[4][c] = zb[7] * gr[3][c];
        }
        for (int a = 0; a < 2; a++)
            for (int b = a + 1; b < 3; b++) {
                const double sm = s2 * (gr[a][b] + gr[b][a]), df = MODELS ? w2 * (gr[a][b] - gr[b][a]) : 0.0;
                o.g[a][b] = sm + df;
                o.g[b][a] = sm - df;
            }
    }
    if (P.nsteady > 0) {
        // - rb[n] nsteady bdf_b fx[n] vol / dt_phy, fx = rho (1, u, v, w, H, ...) - (0, 0, 0, 0, p, ...)
        const double c = -((double)P.nsteady * P.bdf_b * vol / P.dt_phy), rho = d[D_RHO];
        const double e = c * rb[4];
        o.rho += c * rb[0] + e * (d[D_H] + 0.5 * (pc[1] * pc[1] + pc[2] * pc[2] + pc[3] * pc[3]));
        o.h += e * rho;
        o.pc[0] -= e;
        for (int q = 1; q <= 3; q++) {
            o.rho += c * rb[q] * pc[q];
            o.pc[q] += rho * (c * rb[q] + e * pc[q]);
        }
        for (int n = 5; n < NPV; n++) if (n < P.npv) { o.rho += c * rb[n] * pc[n]; o.pc[n] += rho * (c * rb[n]); }
    }
}

// the eddy viscosity's bar mb back to rho, mu, k, omega and the velocity
// gradients through mu_t = sst_eddy_g, one dual pass over (rho, mu, k, omega, S:S)
HD void eddy_back(double mb, const double *pc, const double *d, const double gr[5][3], double ydn, SourceBar &o)
{
    const double x[5] = {d[D_RHO], d[D_MU], pc[7], pc[8], sst_sij<double>(gr[0], gr[1], gr[2])};
    double eb[5];
    dn_grad<5>(5, [&](int q) -> double { return x[q]; },
               [&](auto in, int) -> Dn<5> { return sst_eddy_i<Dn<5>>(in(0), in(1), in(2), in(3), in(4), ydn); }, eb);
    o.rho += mb * eb[0];
    o.mu += mb * eb[1];
    o.pc[7] += mb * eb[2];
    o.pc[8] += mb * eb[3];
    const double s = mb * eb[4];
    for (int a = 0; a < 3; a++) o.g[a][a] += 2.0 * s * gr[a][a];
    for (int a = 0; a < 2; a++)
        for (int b = a + 1; b < 3; b++) {
            const double sm = s * (gr[a][b] + gr[b][a]);
            o.g[a][b] += sm;
            o.g[b][a] += sm;
        }
}

}  // namespace cav

// The reverse passes of 3dcode_amd/csrc/adjoint_point.hpp beside dual-number
// passes of the templated physics they transpose (3dcode_amd/csrc/phys.hpp),
// compiled for the host.  Test infrastructure only.
#include "../../3dcode_amd/csrc/adjoint_point.hpp"

using namespace cav;

extern "C" {

// bars of one variable's 38 stencil points: rev by muscl_back, dual by one-lane passes
void ac_recon(int nlim, int mlp, const double *x, double wl, double wr, double *rev, double *dual)
{
    auto xs = [&](int ll) -> double { return x[ll - 1]; };
    for (int q = 0; q < 38; q++) rev[q] = 0.0;
    const ReconBar r = mlp ? muscl_back<true>(nlim, xs, wl, wr) : muscl_back<false>(nlim, xs, wl, wr);
    const int at[14] = {9, 10, 23, 32, 37, 38, 3, 4, 7, 8, 11, 12, 15, 16};
    const double v[14] = {r.x9, r.x10, r.x23, r.x32, r.x37, r.x38, r.x3, r.x4, r.x7, r.x8, r.x11, r.x12, r.x15, r.x16};
    for (int q = 0; q < 14; q++) rev[at[q] - 1] += v[q];
    if (r.il) rev[r.il - 1] += r.el;
    if (r.ir) rev[r.ir - 1] += r.er;
    for (int q = 0; q < 38; q++) {
        using T = Dn<1>;
        T a, b;
        muscl_var<T>(nlim, mlp != 0, [&](int ll) -> T { return T::seed(x[ll - 1], ll - 1 == q ? 0 : -1); }, a, b);
        dual[q] = wl * a.d[0] + wr * b.d[0];
    }
}

// the ten extrema of the MLP stencil
void ac_extrema(const double *x, double *o)
{
    const MlpExt<double> m = mlp_extrema<double>([&](int ll) -> double { return x[ll - 1]; });
    const double v[10] = {m.ao, m.bo, m.ae, m.be, m.a18, m.b18, m.aL, m.bL, m.aR, m.bR};
    for (int q = 0; q < 10; q++) o[q] = v[q];
}

// flux core of scheme 1 (Roe) or 4 (AUSM+-up): z = {pL[9], pR[9], rhoL, hL, rhoR, hR, c2, u_ref}
void ac_flux(int scheme, int prec, int npv, double pref, double str, const double *n3, const double *z, const double *g,
             double *rev, double *dual)
{
    Par P{};
    P.npv = npv; P.prec = prec; P.pref = pref; P.str = str; P.uref = z[23];
    FaceState<double> L, R;
    for (int n = 0; n < 9; n++) { L.p[n] = z[n]; R.p[n] = z[9 + n]; }
    L.rho = z[18]; L.h = z[19]; R.rho = z[20]; R.h = z[21];
    L.c2 = R.c2 = 0.0;
    FluxBar b;
    if (scheme == 1) roe_back(P, npv, n3, L, R, z[22], g, b);
    else ausm_back(P, npv, n3, L, R, z[22], g, b);
    for (int n = 0; n < 9; n++) { rev[n] = b.pl[n]; rev[9 + n] = b.pr[n]; }
    rev[18] = b.rl; rev[19] = b.hl; rev[20] = b.rr; rev[21] = b.hr; rev[22] = b.c2; rev[23] = b.uref;
    using T = Dn<1>;
    for (int q = 0; q < 24; q++) {
        auto in = [&](int k) { return T::seed(z[k], k == q ? 0 : -1); };
        FaceState<T> l, r;
        for (int n = 0; n < 9; n++) { l.p[n] = in(n); r.p[n] = in(9 + n); }
        l.rho = in(18); l.h = in(19); r.rho = in(20); r.h = in(21); l.c2 = r.c2 = T(0.0);
        Par Pu = P;
        Pu.uref_seed = q == 23 ? 1 : 0;
        const T nt[3] = {T(n3[0]), T(n3[1]), T(n3[2])};
        T fx[NPV], phi(0.0);
        if (scheme == 1) roe_flux<T>(Pu, npv, nt, l, r, in(22), fx);
        else ausm_flux<T>(Pu, npv, nt, l, r, in(22), fx);
        for (int n = 0; n < npv; n++) phi = phi + g[n] * fx[n];
        dual[q] = phi.d[0];
    }
}

// cell properties: sum_m w[m] d[m] back to (p, T, y1, y2); c2: face_c2 alone (w[2] its bar)
void ac_eos(int prop, int c2, const double *x4, const double *w, double *rev, double *dual)
{
    using T = Dn<4>;
    const T p = T::seed(x4[0], 0), t = T::seed(x4[1], 1), y1 = T::seed(x4[2], 2), y2 = T::seed(x4[3], 3);
    T phi(0.0);
    if (c2) {
        c2_back(x4[0], x4[1], x4[2], x4[3], w[D_C2], rev);
        phi = w[D_C2] * face_c2<T>(p, t, y1, y2);
    } else {
        eos_adj(prop != 0, x4, w, rev);
        T d[ND];
        mixture_eos<T>(p, t, y1, y2, d, prop != 0);
        for (int m = 0; m < (prop ? ND : ND - 2); m++) phi = phi + w[m] * d[m];
    }
    for (int q = 0; q < 4; q++) dual[q] = phi.d[q];
}

// viscous flux: z = {g3[6][3], cav[5], muL, kapL, muR, kapR, hTL, hTR, rhoL, rhoR, mutL, mutR}
void ac_visc(int iturb, const double *met, const double *z, const double *g, double *rev, double *dual)
{
    Par P{};
    P.iturb = iturb;
    double e4[4][3], t4[4][3], g3[6][3], dl[ND] = {}, dr[ND] = {};
    const double *n3 = met, *gl = met + 27, *gr = met + 29;
    for (int q = 0; q < 12; q++) { e4[q / 3][q % 3] = met[3 + q]; t4[q / 3][q % 3] = met[15 + q]; }
    for (int q = 0; q < 18; q++) g3[q / 3][q % 3] = z[q];
    dl[D_MU] = z[23]; dl[D_KAP] = z[24]; dr[D_MU] = z[25]; dr[D_KAP] = z[26];
    dl[D_HT] = z[27]; dr[D_HT] = z[28]; dl[D_RHO] = z[29]; dr[D_RHO] = z[30];
    ViscBar b;
    visc_back(P, n3, e4, t4, gl, gr, g3, z + 18, dl, dr, z[31], z[32], g, b);
    for (int q = 0; q < 18; q++) rev[q] = b.g3[q / 3][q % 3];
    for (int q = 0; q < 5; q++) rev[18 + q] = b.cav[q];
    rev[23] = rev[25] = b.mu; rev[24] = rev[26] = b.kap;
    rev[27] = b.ht[0]; rev[28] = b.ht[1]; rev[29] = rev[30] = b.rho; rev[31] = b.mut[0]; rev[32] = b.mut[1];
    using T = Dn<1>;
    for (int q = 0; q < 33; q++) {
        auto in = [&](int k) { return T::seed(z[k], k == q ? 0 : -1); };
        T n[3], e[4][3], t[4][3], l2[2], r2[2], gg[6][3], cv[5], a[ND], c[ND], fx[NPV], phi(0.0);
        for (int k = 0; k < 3; k++) n[k] = T(n3[k]);
        for (int k = 0; k < 12; k++) { e[k / 3][k % 3] = T(e4[k / 3][k % 3]); t[k / 3][k % 3] = T(t4[k / 3][k % 3]); }
        for (int k = 0; k < 2; k++) { l2[k] = T(gl[k]); r2[k] = T(gr[k]); }
        for (int k = 0; k < 18; k++) gg[k / 3][k % 3] = in(k);
        for (int k = 0; k < 5; k++) cv[k] = in(18 + k);
        for (int m = 0; m < ND; m++) { a[m] = T(0.0); c[m] = T(0.0); }
        a[D_MU] = in(23); a[D_KAP] = in(24); c[D_MU] = in(25); c[D_KAP] = in(26);
        a[D_HT] = in(27); c[D_HT] = in(28); a[D_RHO] = in(29); c[D_RHO] = in(30);
        visc_flux<T>(P, n, e, t, l2, r2, gg, cv, a, c, in(31), in(32), fx);
        for (int k = 0; k < (iturb == 0 ? 9 : 7); k++) phi = phi + g[k] * fx[k];
        dual[q] = phi.d[0];
    }
}

}

// source_back and eddy_back of 3dcode_amd/csrc/adjoint_point.hpp beside
// one-lane dual passes over every input of the templated sources
// (3dcode_amd/csrc/phys.hpp), compiled for the host.  Test infrastructure only.
#include "../../3dcode_amd/csrc/adjoint_point.hpp"

using namespace cav;

// inputs: pc 0..8, gradients 9..23, rho 24, h 25, mu 26, mut 27, u_ref 28, dp_ref 29, t_ref 30
static const int NIN = 31;

template <bool MODELS>
static void run(const Par &P, const double *z, const double *d0, const double f6[6][3], double vol, double ydn, const double *rb,
                double mb, double *rev, double *dual)
{
    double d[ND], gr[5][3];
    for (int m = 0; m < ND; m++) d[m] = d0[m];
    for (int q = 0; q < 15; q++) gr[q / 3][q % 3] = z[9 + q];
    SourceBar o;
    source_back<MODELS>(P, z, d, gr, f6, vol, ydn, z[27], rb, o);
    if (mb != 0.0) eddy_back(mb, z, d, gr, ydn, o);
    for (int n = 0; n < 9; n++) rev[n] = o.pc[n];
    for (int q = 0; q < 15; q++) rev[9 + q] = o.g[q / 3][q % 3];
    rev[24] = o.rho; rev[25] = o.h; rev[26] = o.mu; rev[27] = o.mut;
    for (int q = 0; q < 3; q++) rev[28 + q] = o.sc[q];
    using T = Dn<1>;
    for (int q = 0; q < NIN; q++) {
        auto in = [&](int m) { return T::seed(z[m], m == q ? 0 : -1); };
        Par Pu = P;
        Pu.uref_seed = q == 28; Pu.dpref_seed = q == 29; Pu.tref_seed = q == 30;
        T pc[NPV], dt[ND], phi(0.0), g[5][3];
        for (int n = 0; n < NPV; n++) pc[n] = in(n);
        for (int m = 0; m < ND; m++) dt[m] = T(d[m]);
        dt[D_RHO] = in(24); dt[D_H] = in(25); dt[D_MU] = in(26);
        for (int m = 0; m < 15; m++) g[m / 3][m % 3] = in(9 + m);
        if (P.ncav) {
            T rc, rv, ic[4];
            if (MODELS && P.ncav >= 2) {
                T dd[ND], full[18];
                mixture_eos<T>(pc[0] + P.pref, pc[4], pc[5], pc[6], dd, false, full);
                cav_model<T>(Pu, pc, full, vol, rc, rv, ic);
            } else {
                merkle<T>(Pu, pc, dt, vol, rc, rv, ic);
            }
            phi = phi + rb[5] * (rv - rc);
        }
        if (P.iturb == 0) {
            T src[2], it[4], oc;
            sst_source_g<MODELS, T>(P, g[0], g[1], g[2], g[3], g[4], pc[7], pc[8], f6, vol, ydn, dt, in(27), src, it, oc);
            phi = phi + rb[7] * src[0] + rb[8] * src[1];
            if (mb != 0.0) phi = phi + mb * sst_eddy_g<T>(dt[D_RHO], dt[D_MU], pc[7], pc[8], g[0], g[1], g[2], ydn);
        }
        if (P.nsteady > 0) {
            T fx[NPV];
            fx[0] = dt[D_RHO];
            for (int n = 1; n < NPV; n++) fx[n] = dt[D_RHO] * pc[n];
            fx[4] = dt[D_RHO] * (dt[D_H] + 0.5 * (pc[1] * pc[1] + pc[2] * pc[2] + pc[3] * pc[3])) - (pc[0] + P.pref);
            for (int n = 0; n < P.npv; n++) phi = phi - rb[n] * ((double)P.nsteady * (P.bdf_b * fx[n]) * vol / P.dt_phy);
        }
        dual[q] = phi.d[0];
    }
}

extern "C" void sc_source(int models, int ncav, int iturb, int ides, int nsteady, const double *z, const double *d0,
                          const double *f, double vol, double ydn, const double *rb, double mb, double *rev, double *dual)
{
    Par P{};
    P.npv = iturb == 0 ? 9 : 7;
    P.ncav = ncav; P.iturb = iturb; P.ides = ides; P.nsteady = nsteady;
    P.pref = 5.0e3; P.t_crit = 647.0; P.c_c = 0.01; P.c_v = 100.0; P.cav_clip = 1;
    P.uref = z[28]; P.dp_ref = z[29]; P.t_ref = z[30];
    P.bdf_b = 1.5; P.dt_phy = 1e-4;
    double f6[6][3];
    for (int q = 0; q < 18; q++) f6[q / 3][q % 3] = f[q];
    if (models) run<true>(P, z, d0, f6, vol, ydn, rb, mb, rev, dual);
    else run<false>(P, z, d0, f6, vol, ydn, rb, mb, rev, dual);
}

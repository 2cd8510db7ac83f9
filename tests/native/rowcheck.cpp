// The row form of a sweep step (3dcode_amd/csrc/sweep_rows.hpp: the records,
// the stage places, the sixteen lanes of a pencil) on the host, beside the
// row-by-row Jacobian product and D^-1 (jac_apply, getx).  Test infrastructure only.
#include "../../3dcode_amd/csrc/sweep_rows.hpp"
#include <array>
#include <cstring>
#include <vector>

using namespace cav;

namespace {

// The lanes run one after another, a broadcast giving the value its lane had
// in the pass before, until a pass changes none: each pass makes at least one
// more broadcast in the program's order final.
struct Lanes {
    static std::vector<std::array<double, 16>> was, now;
    static int lane_no, call;
    template <int Q> static double lane(double v)
    {
        if (call == (int)was.size()) { was.push_back({}); now.push_back({}); }
        now[call][lane_no] = v;
        return was[call++][Q];
    }
    template <class F> static void run(F f)
    {
        was.clear();
        now.clear();
        for (;;) {
            for (lane_no = 0; lane_no < 16; lane_no++) { call = 0; f(lane_no); }
            if (!memcmp(was.data(), now.data(), was.size() * sizeof(was[0]))) return;
            was = now;
        }
    }
};
std::vector<std::array<double, 16>> Lanes::was, Lanes::now;
int Lanes::lane_no, Lanes::call;

}  // namespace

extern "C" {

// One step: the own cell (0) and its upstream neighbours along i, j, k (1..3).
// cells: 4 x {pv 9, d 13, mut, vol, f6 18}; x: the neighbours' dq; edge: the j
// and k neighbours lie in other tiles.  y, dq by rows of lanes (yr, xr), by
// jac_apply and getx (yp, xp), and by the row coefficients and selections
// that one lane forms alone (ys, xs).
void rc_step(const int *iv, const double *dv, int fwd, int edge, const double *cells, double dt, const double *cc, const double *tt,
             const double *res, const double *x, double *yr, double *xr, double *yp, double *xp, double *ys, double *xs)
{
    Par P{};
    P.npv = iv[0]; P.iturb = iv[2]; P.prec = iv[7]; P.ncav = iv[8]; P.nsteady = iv[9];
    P.cfl = dv[0]; P.pref = dv[1]; P.uref = dv[2]; P.str = dv[3]; P.dt_phy = dv[4]; P.bdf_b = dv[21];
    CellJ c[4];
    double f6[4][6][3], r[4][RC_N];
    for (int q = 0; q < 4; q++) {
        const double *s = cells + 42 * q;
        memcpy(c[q].pv, s, sizeof(c[q].pv));
        memcpy(c[q].d, s + 9, sizeof(c[q].d));
        c[q].mut = s[22]; c[q].vol = s[23];
        memcpy(f6[q], s + 24, sizeof(f6[q]));
        cell_record(P, P.npv, c[q], f6[q], dt, cc, tt, r[q]);
        for (int n = 0; n < NPV; n++) r[q][RC_RES + n] = n < P.npv ? res[n] : 0.0;
    }
    // the parts of a slab: pencils, and the two edge neighbours
    double sp[4][SP_N], se[4][SE_N];
    for (int q = 0; q < 4; q++) {
        for (int e = 0; e < SP_N; e++) sp[q][e] = r[q][stage_item(fwd, e)];
        for (int e = 0; e < SE_N; e++) se[q][e] = q > 0 ? r[q][edge_item(fwd, q - 1, e)] : 0.0;
    }
    Lanes::run([&](int l) {
        const RowMap m = row_map(l, P.npv);
        double k[3][8];
        for (int q = 1; q < 4; q++) {
            const bool e = edge && q > 1;
            row_coef<Lanes>(m, row_jac(jac_at(m, e ? se[q] : sp[q], e, q - 1), 0), k[q - 1]);
        }
        const int ln = l < NPV ? l : 0;
        const RowCell own = row_cell(m, jac_at(m, sp[0], false, 0), sp[0], 0, ln);
        double y = own.res;
        for (int q = 0; q < 3; q++) row_apply<Lanes>(k[q], x[9 * q + ln], y);
        const double v = row_dinv<Lanes>(m, own, y);
        if (l < P.npv) { yr[l] = y; xr[l] = v; }
    });
    const double sgn = fwd ? 1.0 : -1.0;
    const int sign = fwd ? 1 : -1;
    for (int n = 0; n < NPV; n++) yp[n] = ys[n] = n < P.npv ? res[n] : 0.0;
    for (int q = 1; q < 4; q++) {
        const double *n3 = f6[q][2 * (q - 1) + fwd], *xq = x + 9 * (q - 1);
        jac_apply(P, P.npv, c[q], n3, sign, xq, yp, sgn);
        for (int n = 0; n < P.npv; n++) {
            double k[8];
            jac_row_coef(P.npv, jac_nb(c[q].pv, c[q].d, n3, jac_cell(P, c[q]), jac_face(P, c[q], n3), n, P.npv), sign, n, sgn, k);
            jac_row_apply(k, xq, xq[n], ys[n]);
        }
    }
    getx(P, P.npv, c[0], f6[0], dt, cc, tt, yp, xp);
    double g[NGX];
    getx_prep(P, P.npv, c[0], f6[0], dt, cc, tt, g);
    for (int n = 0; n < P.npv; n++)
        xs[n] = getx_apply_sel([&](int q) { return g[q]; }, c[0].pv, c[0].d[D_RY1], c[0].d[D_RT], ys, n, ys[n], c[0].pv[n]);
}

}

// The sweeps' cell records and the row form of a pencil's step.  Host and
// device: X::lane<Q>(v) is v of lane Q of the 16 lanes of a pencil, a DPP
// move in the kernels and stored values in the host tests, which hold these
// functions against jac_apply and getx bit for bit.
#pragma once
#include "phys.hpp"

namespace cav {

// What a sweep step reads of a cell lies side by side in memory, in a record
// of 92 doubles (736 bytes, 46 pieces of 16).  A pencil's records follow one
// another, with a record of zeros before and after each pencil (one between
// two) for the neighbours that it does not have:
//   RC_FP, RC_FM  the +i,+j,+k (-i,-j,-k) faces x (+-n3[3], +-u, lam, vis) / 2:
//                 the forward (backward) sweep's split Jacobians with their
//                 sign and factor (exact: a power of two)
//   RC_Q          the Jacobian's cell terms, in both sweeps
//   RC_GX         the diagonal-inverse terms
//   RC_RES        the residual; the forward sweep puts its dcv there
// Field by field, the sweeps gathered 128 numbers a cell (the shared ones
// once for each of the three pencils that read them) in 32-byte pieces of
// 128-byte lines: 1.46 GB a forward sweep at 128x64x64, sixteen 64-lane
// transfers of 32 lines each a step, whose issue was the length of a step.
// Now it is 86 numbers a cell in whole lines and eleven transfers.
enum { RC_FP = 0, RC_FM = 18, RC_Q = 36, RC_GX = 54, RC_RES = RC_GX + NGX, RC_N = RC_RES + NPV };
enum { Q_RP = 0, Q_RT, Q_RY1, Q_RY2, Q_RHO, Q_BETA, Q_HP, Q_HT, Q_HY1, Q_HY2, Q_U, Q_V, Q_W, Q_Y1, Q_Y2, Q_K, Q_O, Q_H };
static_assert(RC_GX - RC_Q == Q_H + 1 && RC_N == 92, "record layout");

// a cell's record but for its residual
HD void cell_record(const Par &P, int npv, const CellJ &cc, const double f6[6][3], double dt, const double *ic, const double *it, double *__restrict__ r)
{
    for (int q = 0; q < 6; q++) {
        const JacFace f = jac_face(P, cc, f6[q]);
        double *o = r + ((q & 1) ? RC_FP : RC_FM) + 6 * (q >> 1);
        const double h = (q & 1) ? 0.5 : -0.5;
        o[0] = h * f6[q][0]; o[1] = h * f6[q][1]; o[2] = h * f6[q][2];
        o[3] = h * f.u; o[4] = 0.5 * f.lam; o[5] = 0.5 * f.vis;
    }
    const JacCell jc = jac_cell(P, cc);
    double *const c = r + RC_Q;
    c[Q_RP] = cc.d[D_RP]; c[Q_RT] = cc.d[D_RT]; c[Q_RY1] = cc.d[D_RY1]; c[Q_RY2] = cc.d[D_RY2];
    c[Q_RHO] = cc.d[D_RHO]; c[Q_BETA] = jc.beta;
    c[Q_HP] = cc.d[D_HP]; c[Q_HT] = cc.d[D_HT]; c[Q_HY1] = cc.d[D_HY1]; c[Q_HY2] = cc.d[D_HY2];
    c[Q_U] = cc.pv[1]; c[Q_V] = cc.pv[2]; c[Q_W] = cc.pv[3]; c[Q_Y1] = cc.pv[5]; c[Q_Y2] = cc.pv[6];
    c[Q_K] = npv > 7 ? cc.pv[7] : 0.0; c[Q_O] = npv > 7 ? cc.pv[8] : 0.0;
    c[Q_H] = jc.h;
    getx_prep(P, npv, cc, f6, dt, ic, it, r + RC_GX);
}

// A pencil's part of a stage slab (doubles): its cell's F (the sweep's side),
// Q, GX and RES; an edge neighbour's: the F of its face towards the tile, Q
enum { SP_F = 0, SP_Q = 18, SP_GX = 36, SP_RES = SP_GX + NGX, SP_N = SP_RES + NPV, SE_F = 0, SE_Q = 6, SE_N = 24 };
static_assert(SP_N == RC_N - 18 && SP_RES - SP_GX == RC_RES - RC_GX && SP_GX - SP_Q == RC_GX - RC_Q, "stage layout");
// the record's item that stage item q holds; ax: the face's axis
HD int stage_item(bool fwd, int q) { return q + (q < SP_Q ? (fwd ? RC_FP : RC_FM) : RC_Q - SP_Q); }
HD int edge_item(bool fwd, int ax, int q) { return q + (q < SE_Q ? (fwd ? RC_FP : RC_FM) + 6 * ax : RC_Q - SE_Q); }

// Row form of a pencil's step.  A pencil's 16 lanes hold the rows of its
// cell's system; everything else a step reads (the state, properties, face
// and diagonal-inverse terms: some 90 numbers a cell) is the same for all
// lanes.  The lanes read them from the stage one item each (lane l its own
// items, RowMap) and pass them around with DPP row broadcasts.  Reading every
// item into every lane took 140 LDS reads a step, whose return path (each
// read brings 64 lanes x 8 bytes at 128 bytes a clock for the four pencil
// wavefronts of the CU) bound the step.  Now it is 36, and the terms that are
// one expression per column are formed once, a column per lane, not in every
// lane.  What a lane needs another operand for than its neighbours it reads
// from another place rather than selecting among broadcasts.
struct RowMap {
    int v1, a, lb, v2, p, g[7], co[3];     // stage items of this lane, within its pencil's part of a slab
    bool face, aface;               // v1 (and lb), a: items of F (of the i face; the j and k faces' lie 6 and 12 further)
    double one[7];                  // 1 in the lane of the column
    double en, kw, men, mom;        // 1 in lane 4, 1 in the lanes of k and omega, -1 in lane 4, 1 in lanes 1..3
    bool m13, cpl, n0, n4, n5, n7, n8;
};
HD RowMap row_map(int lane, int npv)
{
    RowMap m;
    m.m13 = lane >= 1 && lane <= 3;
    // lanes 0..6: the column's factor of r1 (rho_p, n3, rho_T, rho_y1, rho_y2); lane 13: rho
    m.face = m.m13;
    m.v1 = m.m13 ? SP_F + lane - 1 : SP_Q + (lane == 0 ? Q_RP : lane == 4 ? Q_RT : lane == 5 ? Q_RY1 : lane == 6 ? Q_RY2 : Q_RHO);
    // u, followed by lam and vis; in lanes 1..3 rho
    m.aface = !m.m13;
    m.a = m.m13 ? SP_Q + Q_RHO : SP_F + 3;
    // the factor of lam: in lane 0 beta, else that of u and vis
    m.lb = lane == 0 ? SP_Q + Q_BETA : m.v1;
    // lanes 0..6: the column's factor in the energy row (h_p, u, v, w, h_T, h_y1, h_y2)
    m.v2 = SP_Q + (lane == 0 ? Q_HP : lane <= 3 ? Q_U + lane - 1 : lane == 4 ? Q_HT : lane == 5 ? Q_HY1 : Q_HY2);
    // the row's own factor: pv(n), in the energy row the total enthalpy
    // (lane 0 and the lanes without a row read one that they do not use)
    m.p = SP_Q + (m.m13 ? Q_U + lane - 1 : lane == 4 ? Q_H : lane >= 5 && lane <= 8 ? Q_Y1 + lane - 5 : Q_U);
    // the row's entries of D^-1 (getx_apply): k1..k4, e1, e2, f1
    m.n0 = lane == 0; m.n4 = lane == 4; m.n5 = lane == 5; m.n7 = lane == 7; m.n8 = lane == 8;
    m.cpl = m.n0 || m.n4 || m.n5;
    const bool row7 = lane >= 7;
    m.g[0] = SP_GX + (m.n0 ? GX_C4C1 : m.n4 ? GX_C4IB1S1 : m.n7 ? GX_RBT4 : m.n8 ? GX_RBT1 : GX_C4SSIB1);
    m.g[1] = SP_GX + (m.n0 ? GX_C2 : m.n4 ? GX_C1 : m.n7 ? GX_T2 : m.n8 ? GX_T3 : GX_SS);
    m.g[2] = SP_GX + (m.n0 ? GX_C3 : m.n4 ? GX_C3IB1 : GX_C1);
    m.g[3] = SP_GX + (m.n0 ? GX_RB1 : GX_C2IB1);
    m.g[4] = SP_GX + (m.n0 ? GX_CROSS1 : GX_S1P5);
    m.g[5] = SP_GX + (m.n0 ? GX_CP5 : GX_SSY1);
    m.g[6] = SP_GX + (m.cpl ? GX_MM : row7 ? GX_IT : GX_IB1);
    // lanes 0, 1, 2: the three sums res0 a + b uuu + c res6 that rows 0, 4, 5 share
    m.co[0] = SP_GX + (lane == 0 ? GX_AAA1 : lane == 1 ? GX_AAA2 : GX_SSHM);
    m.co[1] = lane == 0 ? SP_Q + Q_RY1 : lane == 1 ? SP_Q + Q_RT : SP_GX + GX_RRR;
    m.co[2] = SP_GX + (lane == 0 ? GX_CROSS : lane == 1 ? GX_CROSS2 : GX_SSY2);
    for (int l = 0; l < 7; l++) m.one[l] = lane == l ? 1.0 : 0.0;
    m.en = m.one[4]; m.men = -m.one[4];
    m.mom = m.m13 ? 1.0 : 0.0;
    m.kw = row7 && lane < npv ? 1.0 : 0.0;
    return m;
}

// A lane's Jacobian items of a cell and face (RowMap): v1, u (rho in lanes
// 1..3), lam, vis, the factor of lam, v2, p
struct RowJac {
    double v1, a, b, c, lb, v2, p;
};
// where they lie: of the part st of a slab (an edge neighbour's or a
// pencil's), the face of axis ax; and their values in the slab that starts
// `slab` further
struct JacAt { const double *v1, *a, *lb, *v2, *p; };
HD JacAt jac_at(const RowMap &m, const double *st, bool edge, int ax)
{
    const int q = edge ? SE_Q - SP_Q : 0, f = edge ? 0 : 6 * ax;
    return JacAt{st + m.v1 + (m.face ? f : q), st + m.a + (m.aface ? f : q), st + m.lb + (m.face ? f : q), st + m.v2 + q, st + m.p + q};
}
HD RowJac row_jac(const JacAt &w, int slab)
{
    return RowJac{w.v1[slab], w.a[slab], w.a[slab + 1], w.a[slab + 2], w.lb[slab], w.v2[slab], w.p[slab]};
}

// Row coefficients of one neighbour's split Jacobian, c[l] = +-0.5 a(n,l)
// (jac_row's products and sums in its order; jac_row_coef has the same row by
// row): r1[l] and the energy row's factor of column l sit in lane l.  The
// factor 0.5 and the sign are in u, lam, vis and n3 already, which they pass
// through exactly.  A term that only some rows have is added as
// fma(term, 1 or 0, sum), which rounds as the sum where the term is finite.
// A term that is not makes NaN of the rows that do not have it; those are
// not finite without it either (u, lam or vis are in every row's columns), so
// a run that overflows loses the same rows and only shows NaN where
// jac_row_coef shows infinity.  (Selecting the term takes three instructions
// for each fma.)
template <class X> HD void row_coef(const RowMap &m, const RowJac &j, double *c)
{
    const double t0 = j.a * j.v1, t = t0 + j.b * j.lb + j.c * j.v1, r = m.m13 ? t0 : t;
    // (lane 13 holds rho, u, lam and vis; the broadcasts stay out of the
    // selects: they need every lane active)
    const double ru = X::template lane<13>(j.v1 * (j.a + j.b + j.c));
    const double P = m.n0 ? 1.0 : j.p, Q = ru * m.en;
    c[0] = P * X::template lane<0>(r) + Q * X::template lane<0>(j.v2);
    c[1] = P * X::template lane<1>(r) + Q * X::template lane<1>(j.v2);
    c[2] = P * X::template lane<2>(r) + Q * X::template lane<2>(j.v2);
    c[3] = P * X::template lane<3>(r) + Q * X::template lane<3>(j.v2);
    c[4] = P * X::template lane<4>(r) + Q * X::template lane<4>(j.v2);
    c[5] = P * X::template lane<5>(r) + Q * X::template lane<5>(j.v2);
    c[6] = P * X::template lane<6>(r) + Q * X::template lane<6>(j.v2);
    // the pressure column: n3 in the momentum rows, -lam, then -vis in the energy row
    c[0] = fma(j.v1, m.mom, c[0]);
    c[0] = fma(j.b, m.men, c[0]);
    c[0] = fma(j.c, m.men, c[0]);
#pragma unroll
    for (int l = 1; l < 7; l++) if (l != 4) c[l] = fma(ru, m.one[l], c[l]);
    c[7] = ru * m.kw;
}

// y += c x, the neighbour's row n in lane n (jac_row_apply)
template <class X> HD void row_apply(const double *c, double x, double &y)
{
    y = y + c[0] * X::template lane<0>(x);
    y = y + c[1] * X::template lane<1>(x);
    y = y + c[2] * X::template lane<2>(x);
    y = y + c[3] * X::template lane<3>(x);
    y = y + c[4] * X::template lane<4>(x);
    y = y + c[5] * X::template lane<5>(x);
    y = y + c[6] * X::template lane<6>(x);
    y = y + c[7] * x;
}

// What a step reads of its own cell, read during the step before: the rows'
// residual, the Jacobian items, the rows' D^-1 entries
struct RowCell {
    RowJac j;
    double res, g[7], a, co[3];
};
// ln: the lane's row, 0 where it has none
HD RowCell row_cell(const RowMap &m, const JacAt &at, const double *st, int slab, int ln)
{
    RowCell c;
    c.j = row_jac(at, slab);
    c.res = st[slab + SP_RES + ln];
#pragma unroll
    for (int q = 0; q < 7; q++) c.g[q] = st[slab + m.g[q]];
    c.a = st[slab + SP_GX + GX_A];
#pragma unroll
    for (int q = 0; q < 3; q++) c.co[q] = st[slab + m.co[q]];
    return c;
}

// Row n of D^-1 y in lane n (y: the row's right-hand side).  Rows 0, 4 and 5
// are sums of four products, rows 7 and 8 of two, the rest one difference:
// every row forms ((k1 x1 + k2 x2) + k3 x3) + k4 ((x4 + e1 z1) + e2 z2) with
// its own entries and operands and takes the partial sum it needs.
// Subtractions are sums with the entry's sign flipped, so the operations and
// their order are getx_apply's.
template <class X> HD double row_dinv(const RowMap &m, const RowCell &c, double y)
{
    auto neg = [](double x, bool f) {
        return __builtin_bit_cast(double, __builtin_bit_cast(unsigned long long, x) ^ ((unsigned long long)f << 63));
    };
    const double y0 = X::template lane<0>(y), y5 = X::template lane<5>(y), y6 = X::template lane<6>(y);
    const double s1 = y - y0 * c.j.p;
    const double r6 = X::template lane<6>(s1), rk = X::template lane<7>(s1), ro = X::template lane<8>(s1);
    const double uuu = X::template lane<1>(y) * X::template lane<1>(c.j.v2) + X::template lane<2>(y) * X::template lane<2>(c.j.v2)
                     + X::template lane<3>(y) * X::template lane<3>(c.j.v2) - X::template lane<4>(y);
    const double co = y0 * c.co[0] + c.co[1] * uuu + c.co[2] * y6;
    const double co1 = X::template lane<0>(co), co2 = X::template lane<1>(co), co3 = X::template lane<2>(co);
    const bool row7 = m.n7 || m.n8;
    const double x1 = row7 ? s1 : r6;
    const double x2 = m.n5 ? s1 : m.n7 ? ro : m.n8 ? rk : co1;
    const double x3 = m.n4 ? co3 : co2, x4 = m.n0 ? co2 : co3;
    const double z1 = m.n0 ? y5 : y0, z2 = m.n0 ? y0 : y5;
    const double s2 = neg(c.g[0], !m.n4) * x1 + neg(c.g[1], m.n0) * x2;
    const double w = x4 + neg(c.g[4], !m.n0) * z1 + neg(c.g[5], m.n0) * z2;
    const double s4 = s2 + neg(c.g[2], !m.n0) * x3 + (m.n4 ? -1.0 : c.g[3]) * (m.n5 ? x4 : w);
    return (m.cpl ? s4 : row7 ? s2 : s1) * c.g[6] * c.a;
}

}  // namespace cav

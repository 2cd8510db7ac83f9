// Discrete adjoint of the residual: cav3d_rhs_vjp.
//
// The operator is the residual cav3d_calrhs evaluates (src/rhs_module.f90:
// 260-643: inviscid and viscous face-flux differences, the mass-transfer and SST
// sources, the BDF term), taken as a function of every block's ghosted
// primitive state pv, with the cell properties re-derived from pv by the EOS
// (rho, h, c^2, the EOS derivatives, mu, kappa: deteos_prop) and with the
// eddy viscosity, the grid metrics, the BDF history and the ghost layers
// held fixed (a ghost cell is an input like an interior cell).  It returns
//   pv_bar = (d res / d pv)^T res_bar
// and the two scalar derivatives of res_bar . res with respect to p_ref and
// u_ref.  The reference has no adjoint; this is the VJP of its residual.
//
// Method: reverse accumulation over faces and cells.  Each face recomputes its
// reconstruction and flux (nothing is kept from a forward pass) and runs them
// backwards from g_f = res_bar(right cell) - res_bar(left cell)
// (adjoint_point.hpp), leaving the bars of its two reconstructed states and
// of its viscous differences.  A stencil pass (k_adj_stencil) then takes those
// through the reconstruction and the differences to the stencil points, one
// wavefront per tile of cells and variable: it runs every face whose stencil
// reaches its cells, in a fixed order, and adds what falls on them in LDS, so
// no bars of stencil points are written to memory and the result is
// deterministic.  The cell sources are differentiated per cell (dual passes over
// the few numbers each source reads), and each cell's property bars return to (p, T, y1, y2) through its
// EOS.  Arithmetic is FP64 throughout.
//
// d/d(p_ref) is the sum of pv_bar over the pressure component: the residual
// reads gauge pressure only as p + p_ref or in differences (the pressure
// floor included), so shifting p_ref shifts it as shifting every gauge
// pressure does.  d/d(u_ref) comes out of the flux cores' reverse passes (the
// low-Mach preconditioning is its only reader there) and of the mass-transfer
// sources'.
//
// Included once, from cav3d.hip, after the context definition.

#include "adjoint_point.hpp"

namespace {

struct AD {
    const double *rb;       // res_bar [npv][NC]
    double *w[3];           // a face's reconstruction bars [2][npv][NF]: left, right
    int *cell[3];           // which of them belong to the cells' own values (FaceBar::cell) [NF]
    double *snb[3];         // a face's sensor-pressure bars [18][NF] (Roe-M, AUSMPW+)
    double *fp[3];          // first-order faces: bars of rho, h, c^2 of the two cells [2][3][NF]
    double *vb[3];          // a face's viscous bars [3 nv + ncv][NF]: differences, averages
    double *vp[3];          // and of its cells' properties [5][NF]: mu, kappa, rho (each side), h_T left, right
    double *ub[3];          // d(phi_f)/d(u_ref) [NF]
    double *cb;             // cell-source bars [npv (+ 15)][NC]: of the cell's state, and under SST of its
                            // gradients of u, v, w, k, omega (half of them, over the volume)
    double *cdb;            // cell-source property bars [3][NC]: rho, h, mu
    double *csb;            // cell-source d(phi_c)/d(u_ref, dp_ref, t_ref) [3][NC] (the mass-transfer scales)
    double *pb;             // pv_bar [npv][NG]
    double *pbd[3];         // the stencil pass's share of it, by direction
    double *mtb[3];         // eddy-viscosity bars of a face's two cells [2][NF] (dmut)
    const int *tiles[3];    // tiles of the stencil pass by direction: block, first i, j, k
    int ntiles[3];
    int dmut;               // 1: the interior cells' eddy viscosity is the SST function of
                            // the state (differentiated); 0: held fixed
};

__device__ __forceinline__ bool interior_cell(const BlkD &B, int i, int j, int k)
{
    return i >= 2 && i <= B.I && j >= 2 && j <= B.J && k >= 2 && k <= B.K;
}

__device__ __forceinline__ double rbar(const DS &S, const AD &A, const BlkD &B, int i, int j, int k, int n)
{
    return interior_cell(B, i, j, k) ? A.rb[(long)n * S.NC + cidx(B, i, j, k)] : 0.0;
}

// (normal, first transverse, second transverse) offset of stencil point ll
// from the face's left cell; the same table as stencil_off
__device__ __forceinline__ void stencil_ijk(int ll, int &dn, int &de, int &dt)
{
    int q = ll - 1;
    if (q < 18) { dn = q & 1; de = (q >> 1) % 3 - 1; dt = q / 6 - 1; }
    else if (q < 27) { q -= 18; dn = -1; de = q % 3 - 1; dt = q / 3 - 1; }
    else if (q < 36) { q -= 27; dn = 2; de = q % 3 - 1; dt = q / 3 - 1; }
    else { dn = q == 36 ? -2 : 3; de = 0; dt = 0; }
}

// does the face of direction D with left cell (i,j,k) exist
__device__ __forceinline__ bool face_exists(const BlkD &B, int D, int i, int j, int k)
{
    const int lo[3] = {D == 0 ? 1 : 2, D == 1 ? 1 : 2, D == 2 ? 1 : 2};
    return i >= lo[0] && i <= B.I && j >= lo[1] && j <= B.J && k >= lo[2] && k <= B.K;
}

// Inviscid part of a face up to its reconstruction: the bars of its left and
// right states (k_adj_stencil takes them to the stencil points), the cells'
// property bars (first order) and the u_ref derivative.
template <int D, bool SENSOR>
__device__ __forceinline__ void face_vjp(const DS &S, const AD &A, unsigned wg)
{
    long t = (long)wg * blockDim.x + threadIdx.x;
    if (t >= S.NF[D]) return;
    int i, j, k;
    const BlkD &B = face_of<D>(S, t, i, j, k);
    const Par &P = S.P;
    const int npv = S.npv;
    const long NF = S.NF[D];
    const long g9 = gidx(B, i, j, k);
    const long sN = D == 0 ? 1 : (D == 1 ? (long)B.nx : (long)B.nx * B.ny);
    const long gq = g9 + sN;
    const int ip = i + (D == 0), jp = j + (D == 1), kp = k + (D == 2);
    double g[NPV];
    bool any = false;
    for (int n = 0; n < NPV; n++) {
        g[n] = n < npv ? rbar(S, A, B, ip, jp, kp, n) - rbar(S, A, B, i, j, k, n) : 0.0;
        any = any || g[n] != 0.0;
    }
    FaceBar o;
    if (any) {
        const double *f0 = S.pv + g9;
        double n3[3];
        face_vec(S, B, D, i, j, k, n3);
        const double cellp[6] = {S.dc[D_RHO * S.NG + g9], S.dc[D_H * S.NG + g9], S.dc[D_C2 * S.NG + g9],
                                 S.dc[D_RHO * S.NG + gq], S.dc[D_H * S.NG + gq], S.dc[D_C2 * S.NG + gq]};
        face_adj_core<SENSOR>(P, npv, [&](int ll, int n) -> double { return f0[(long)n * S.NG + stencil_off<D>(B, ll)]; },
                              n3, cellp, g, o);
    } else {
        for (int n = 0; n < NPV; n++) o.wl[n] = o.wr[n] = 0.0;
        for (int q = 0; q < 18; q++) o.sen[q] = 0.0;
        for (int q = 0; q < 3; q++) o.prop[0][q] = o.prop[1][q] = 0.0;
        o.uref = 0.0;
        o.cell = 0;
    }
    for (int n = 0; n < NPV; n++) if (n < npv) {
        A.w[D][(long)n * NF + t] = o.wl[n];
        A.w[D][(long)(npv + n) * NF + t] = o.wr[n];
    }
    A.cell[D][t] = o.cell;
    if (SENSOR) for (int q = 0; q < 18; q++) A.snb[D][q * NF + t] = o.sen[q];
    if (P.nmuscl == 0)
        for (int q = 0; q < 3; q++) {
            A.fp[D][q * NF + t] = o.prop[0][q];
            A.fp[D][(3 + q) * NF + t] = o.prop[1][q];
        }
    A.ub[D][t] = o.uref;
}

// Viscous part of a face: the bars of its differences and averages (linear in
// the stencil, k_adj_stencil applies them), of the two cells' mu, kappa and,
// under SST, rho, h_T and eddy viscosity.
template <int D>
__device__ __forceinline__ void vface_vjp(const DS &S, const AD &A, unsigned wg)
{
    long t = (long)wg * blockDim.x + threadIdx.x;
    if (t >= S.NF[D]) return;
    int i, j, k;
    const BlkD &B = face_of<D>(S, t, i, j, k);
    const Par &P = S.P;
    const int npv = S.npv;
    const long NF = S.NF[D];
    const long g9 = gidx(B, i, j, k);
    const long sN = D == 0 ? 1 : (D == 1 ? (long)B.nx : (long)B.nx * B.ny);
    const long gq = g9 + sN;
    int ip = i, jp = j, kp = k;
    if (D == 0) ip++; else if (D == 1) jp++; else kp++;
    double gf[NPV];
    for (int n = 0; n < NPV; n++) gf[n] = n < npv ? rbar(S, A, B, i, j, k, n) - rbar(S, A, B, ip, jp, kp, n) : 0.0;
    const bool turb = P.iturb == 0;
    const int nv = turb ? 6 : 4, ncv = turb ? 5 : 3;
    // inputs: the normal / transverse differences, the face averages, the cell properties
    double g3[6][3], cav[5];
#pragma unroll
    for (int q = 0; q < 6; q++) {
        const int n = q < 4 ? q + 1 : q + 3;
        if (q >= nv) { g3[q][0] = g3[q][1] = g3[q][2] = 0.0; continue; }
        auto xs = [&](int ll) -> double { return S.pv[(long)n * S.NG + g9 + stencil_off<D>(B, ll)]; };
        g3[q][0] = xs(10) - xs(9);
        g3[q][1] = 0.0625 * (-xs(1) - xs(2) + xs(5) + xs(6) + 2.0 * (-xs(7) - xs(8) + xs(11) + xs(12)) - xs(13) - xs(14) + xs(17) + xs(18));
        g3[q][2] = 0.0625 * (-xs(1) - xs(2) + xs(13) + xs(14) + 2.0 * (-xs(3) - xs(4) + xs(15) + xs(16)) - xs(5) - xs(6) + xs(17) + xs(18));
        if (q < 3) cav[q] = 0.5 * (xs(9) + xs(10));
        if (q > 3) cav[q - 1] = 0.5 * (xs(9) + xs(10));
    }
    if (!turb) cav[3] = cav[4] = 0.0;
    double dl[ND], dr[ND];
    for (int m = 0; m < ND; m++) { dl[m] = S.dc[m * S.NG + g9]; dr[m] = S.dc[m * S.NG + gq]; }
    const double ml = S.mut ? S.mut[g9] : 0.0, mr = S.mut ? S.mut[gq] : 0.0;
    // metrics (as visc_face)
    double n3[3], e4[4][3], t4[4][3];
    face_vec(S, B, D, i, j, k, n3);
    const int E = (D + 1) % 3, T = (D + 2) % 3;
    int p0[3] = {i, j, k}, p1[3] = {ip, jp, kp};
    int a0[3], a1[3];
    for (int q = 0; q < 3; q++) { a0[q] = p0[q]; a1[q] = p1[q]; }
    a0[E]--; a1[E]--;
    face_vec(S, B, E, a0[0], a0[1], a0[2], e4[0]);
    face_vec(S, B, E, a1[0], a1[1], a1[2], e4[1]);
    face_vec(S, B, E, p0[0], p0[1], p0[2], e4[2]);
    face_vec(S, B, E, p1[0], p1[1], p1[2], e4[3]);
    for (int q = 0; q < 3; q++) { a0[q] = p0[q]; a1[q] = p1[q]; }
    a0[T]--; a1[T]--;
    face_vec(S, B, T, a0[0], a0[1], a0[2], t4[0]);
    if (D == 0) {
        face_vec(S, B, T, a1[0], a1[1], a1[2], t4[1]);
        face_vec(S, B, T, p0[0], p0[1], p0[2], t4[2]);
    } else {
        face_vec(S, B, T, p0[0], p0[1], p0[2], t4[1]);
        face_vec(S, B, T, a1[0], a1[1], a1[2], t4[2]);
    }
    face_vec(S, B, T, p1[0], p1[1], p1[2], t4[3]);
    const long wl = widx(B, i, j, k), wr = widx(B, ip, jp, kp);
    const double gl[2] = {S.vol[wl], S.ydn ? S.ydn[wl] : 1.0}, gr[2] = {S.vol[wr], S.ydn ? S.ydn[wr] : 1.0};
    ViscBar o;
    visc_back(P, n3, e4, t4, gl, gr, g3, cav, dl, dr, ml, mr, gf, o);
    double *vb = A.vb[D], *vp = A.vp[D];
#pragma unroll
    for (int q = 0; q < 6; q++) if (q < nv) for (int c = 0; c < 3; c++) vb[(long)(3 * q + c) * NF + t] = o.g3[q][c];
#pragma unroll
    for (int q = 0; q < 5; q++) if (q < ncv) vb[(long)(3 * nv + q) * NF + t] = o.cav[q];
    vp[t] = o.mu;
    vp[NF + t] = o.kap;
    if (turb) {
        vp[2 * NF + t] = o.rho;
        vp[3 * NF + t] = o.ht[0];
        vp[4 * NF + t] = o.ht[1];
        if (A.dmut) { A.mtb[D][t] = o.mut[0]; A.mtb[D][NF + t] = o.mut[1]; }
    }
}

// Every face's bars in one launch, the directions' inviscid parts and then
// their viscous ones, as k_face (all of them run one wavefront per SIMD).
template <bool SENSOR>
__global__ __launch_bounds__(128) void k_faces_vjp(DS S, AD A, FluxWgs g)
{
    unsigned w = blockIdx.x;
    if (w < g.n[0]) { face_vjp<0, SENSOR>(S, A, w); return; }
    w -= g.n[0];
    if (w < g.n[1]) { face_vjp<1, SENSOR>(S, A, w); return; }
    w -= g.n[1];
    if (w < g.n[2]) { face_vjp<2, SENSOR>(S, A, w); return; }
    w -= g.n[2];
    if (w < g.n[0]) { vface_vjp<0>(S, A, w); return; }
    w -= g.n[0];
    if (w < g.n[1]) { vface_vjp<1>(S, A, w); return; }
    vface_vjp<2>(S, A, w - g.n[1]);
}

// The stencil pass: one wavefront owns a tile of ghosted cells, one variable
// and one direction, and adds to the tile, in LDS, what every face of that
// direction whose stencil reaches it leaves on its points: the reconstruction run
// backwards from the face's two bars (muscl_back) and the viscous differences'
// transposes.  Faces near a tile's edge are run by every tile they reach,
// which costs arithmetic but no memory: with the bars of all 38 points written
// per face and variable and gathered by a second kernel, a product moved 9 GB
// through them at 128 x 64 x 64.  A stencil reaches further along its normal
// (-2 .. 3) than across (-1 .. 1), so a direction's tile (16 KB of LDS) is
// twice as long along it: 1.8 runs a face, 2.2 with one 16 x 8 x 8 tile for
// the three directions.  SMALL: 16 x 8 x 8, for grids with too few of the
// larger tiles to fill the chip (adj_alloc).  Within one LDS add the lanes (distinct faces, one
// stencil point) hit distinct cells, and a wavefront's LDS operations run in
// its program order, so the sums have a fixed order.
// What bounds it: the arithmetic of the reconstruction's bound and its
// transpose (780 vector instructions a round of 64 faces) at two
// wavefronts a SIMD, which the 38 stencil values in registers allow; three
// spill (1.95 -> 2.43 ms).  128x64x64 cells, MLP, nine variables: 2.6 ms with
// one tile for the three directions and a selected extremum looped over, 1.95
// with the limiter's bars in registers, 1.58 with a tile a direction.
constexpr int ADJ_TILE[2][3][3] = {{{32, 8, 8}, {16, 16, 8}, {16, 8, 16}}, {{16, 8, 8}, {16, 8, 8}, {16, 8, 8}}};
constexpr int ADJ_CELLS[2] = {2048, 1024};
template <int D, int NM, bool SMALL>
__device__ __forceinline__ void adj_stencil_dir(const DS &S, const AD &A, int item, double *acc)
{
    constexpr int TI = ADJ_TILE[SMALL][D][0], TJ = ADJ_TILE[SMALL][D][1], TK = ADJ_TILE[SMALL][D][2], NT = TI * TJ * TK;
    static_assert(NT == ADJ_CELLS[SMALL], "a tile fills the LDS array");
    const int n = item / A.ntiles[D];
    const int *td = A.tiles[D] + 4 * (item - n * A.ntiles[D]);
    const BlkD &B = S.b[td[0]];
    const int c0[3] = {td[1], td[2], td[3]};
    const int c1[3] = {min(c0[0] + TI - 1, B.I + 3), min(c0[1] + TJ - 1, B.J + 3), min(c0[2] + TK - 1, B.K + 3)};
    for (int q = threadIdx.x; q < NT; q += 64) acc[q] = 0.0;
    const bool visc = S.P.iturb >= -2;
    // the variable's place among the viscous differences (u, v, w, T, k, omega) and averages (u, v, w, k, omega)
    const int vq = !visc ? -1 : (n >= 1 && n <= 4) ? n - 1 : n >= 7 ? n - 3 : -1;
    const int cq = !visc ? -1 : (n >= 1 && n <= 3) ? n - 1 : n >= 7 ? n - 4 : -1;
    const int nv = S.P.iturb == 0 ? 6 : 4;
    const double *sen = n == 0 && (S.P.nscheme == 2 || S.P.nscheme == 3) ? A.snb[D] : nullptr;
    constexpr int E = (D + 1) % 3, T = (D + 2) % 3;
    const int npv = S.npv, ext[3] = {B.I, B.J, B.K}, lane = threadIdx.x;
    const long NF = S.NF[D];
    int lo[3], cnt[3];
    lo[D] = max(c0[D] - 3, 1);
    lo[E] = max(c0[E] - 1, 2);
    lo[T] = max(c0[T] - 1, 2);
    cnt[D] = min(c1[D] + 2, ext[D]) - lo[D] + 1;
    cnt[E] = min(c1[E] + 1, ext[E]) - lo[E] + 1;
    cnt[T] = min(c1[T] + 1, ext[T]) - lo[T] + 1;
    // (no face reaches a tile that lies beyond the last ghost layer but one)
    const int total = cnt[0] > 0 && cnt[1] > 0 && cnt[2] > 0 ? cnt[0] * cnt[1] * cnt[2] : 0;
    constexpr int st[3] = {1, TI, TI * TJ};
    const int fn[2] = {D == 0 ? B.I : B.I - 1, D == 1 ? B.J : B.J - 1};       // the block's faces along i and j
    // q / cnt of small numbers through the reciprocal: (q + 0.5) / cnt is at
    // least 0.5 / cnt away from every whole number, far more than it is rounded by
    const float i0 = 1.0f / (float)cnt[0], i1 = 1.0f / (float)cnt[1];
    for (int base = 0; base < total; base += 64) {
        const int r = base + lane;
        const bool on = r < total;
        const int q = on ? r : 0;
        const int q1 = (int)(((float)q + 0.5f) * i0), q2 = (int)(((float)q1 + 0.5f) * i1);
        const int f[3] = {lo[0] + q - q1 * cnt[0], lo[1] + q1 - q2 * cnt[1], lo[2] + q2};
        // the face's place in its block (fidx)
        const unsigned t = (unsigned)(f[0] - (D == 0 ? 1 : 2) + fn[0] * (f[1] - (D == 1 ? 1 : 2) + fn[1] * (f[2] - (D == 2 ? 1 : 2))));
        double wl = at32(A.w[D] + (long)n * NF + B.f0[D], t), wr = at32(A.w[D] + (long)(npv + n) * NF + B.f0[D], t);
        const int cell = at32(A.cell[D] + B.f0[D], t);
        // the face's left cell in tile coordinates; which offsets along each axis land in the tile
        const int l[3] = {f[0] - c0[0], f[1] - c0[1], f[2] - c0[2]};
        const int w3[3] = {c1[0] - c0[0], c1[1] - c0[1], c1[2] - c0[2]};
        bool inN[6], inE[3], inT[3];
#pragma unroll
        for (int d = 0; d < 6; d++) inN[d] = on && (unsigned)(l[D] + d - 2) <= (unsigned)w3[D];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            inE[d] = (unsigned)(l[E] + d - 1) <= (unsigned)w3[E];
            inT[d] = (unsigned)(l[T] + d - 1) <= (unsigned)w3[T];
        }
        const int at = l[0] * st[0] + l[1] * st[1] + l[2] * st[2];
        auto add = [&](int ll, double v) {
            int dn, de, dt;
            stencil_ijk(ll, dn, de, dt);
            if (inN[dn + 2] && inE[de + 1] && inT[dt + 1])
                __hip_atomic_fetch_add(&acc[at + dn * st[D] + de * st[E] + dt * st[T]], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        const bool cl = NM == 0 || ((cell >> n) & 1), cr = NM == 0 || ((cell >> (16 + n)) & 1);
        double b9 = cl ? wl : 0.0, b10 = cr ? wr : 0.0;
        wl = cl ? 0.0 : wl;
        wr = cr ? 0.0 : wr;
        ReconBar o;
        o.x9 = o.x10 = o.x23 = o.x32 = o.x37 = o.x38 = 0.0;
        o.x3 = o.x4 = o.x7 = o.x8 = o.x11 = o.x12 = o.x15 = o.x16 = o.el = o.er = 0.0;
        o.il = o.ir = 0;
        // the viscous bars and the stencil, read ahead of the arithmetic (and
        // whether or not the reconstruction's bars are zero): one memory latency a round
        double v0 = 0.0, v1 = 0.0, v2 = 0.0, vc = 0.0;
        if (vq >= 0) {
            v0 = at32(A.vb[D] + (long)(3 * vq) * NF + B.f0[D], t);
            v1 = 0.0625 * at32(A.vb[D] + (long)(3 * vq + 1) * NF + B.f0[D], t);
            v2 = 0.0625 * at32(A.vb[D] + (long)(3 * vq + 2) * NF + B.f0[D], t);
            if (cq >= 0) vc = 0.5 * at32(A.vb[D] + (long)(3 * nv + cq) * NF + B.f0[D], t);
        }
        if constexpr (NM > 0) {
            const double *f0 = S.pv + (long)n * S.NG + B.g0;
            const unsigned gl = (unsigned)(f[0] + 1 + B.nx * (f[1] + 1 + B.ny * (f[2] + 1)));
            double x[NSLOT];
#pragma unroll
            for (int ll = 1; ll <= NSLOT; ll++)
                if (NM == 2 || ll == 9 || ll == 10 || ll == 23 || ll == 32 || ll >= 37) x[ll - 1] = at32(f0 + stencil_off<D>(B, ll), gl);
            if (on && (wl != 0.0 || wr != 0.0)) o = muscl_back<NM == 2>(S.P.nlim, [&](int ll) -> double { return x[ll - 1]; }, wl, wr);
        }
        b9 += o.x9;
        b10 += o.x10;
        // the bar of the extremum a side's MLP bound selected, if that is point ll
        auto exl = [&](int ll) -> double { return NM == 2 && o.il == ll ? o.el : 0.0; };
        auto exr = [&](int ll) -> double { return NM == 2 && o.ir == ll ? o.er : 0.0; };
        auto ex = [&](int ll) -> double { return exl(ll) + exr(ll); };
        if (vq >= 0 || sen) {
            // the 18 points of the viscous differences (and of the pressure sensor)
            auto sn = [&](int ll) -> double { return (sen ? at32(sen + (long)(ll - 1) * NF + B.f0[D], t) : 0.0) + ex(ll); };
            add(1, -v1 - v2 + sn(1));
            add(2, -v1 - v2 + sn(2));
            add(3, o.x3 - 2.0 * v2 + sn(3));
            add(4, o.x4 - 2.0 * v2 + sn(4));
            add(5, v1 - v2 + sn(5));
            add(6, v1 - v2 + sn(6));
            add(7, o.x7 - 2.0 * v1 + sn(7));
            add(8, o.x8 - 2.0 * v1 + sn(8));
            add(9, b9 + vc - v0 + sn(9));
            add(10, b10 + vc + v0 + sn(10));
            add(11, o.x11 + 2.0 * v1 + sn(11));
            add(12, o.x12 + 2.0 * v1 + sn(12));
            add(13, -v1 + v2 + sn(13));
            add(14, -v1 + v2 + sn(14));
            add(15, o.x15 + 2.0 * v2 + sn(15));
            add(16, o.x16 + 2.0 * v2 + sn(16));
            add(17, v1 + v2 + sn(17));
            add(18, v1 + v2 + sn(18));
        } else {
            add(9, b9 + ex(9));
            add(10, b10 + ex(10));
            if constexpr (NM == 2) {
                add(3, o.x3 + ex(3)); add(4, o.x4 + ex(4)); add(7, o.x7 + ex(7)); add(8, o.x8 + ex(8));
                add(11, o.x11 + ex(11)); add(12, o.x12 + ex(12)); add(15, o.x15 + ex(15)); add(16, o.x16 + ex(16));
                auto corner = [&](int ll) { if (o.il == ll || o.ir == ll) add(ll, ex(ll)); };
                corner(1); corner(2); corner(5); corner(6); corner(13); corner(14); corner(17); corner(18);
            }
        }
        if constexpr (NM > 0) {
            add(23, o.x23 + exl(23));
            add(32, o.x32 + exr(32));
            add(37, o.x37);
            add(38, o.x38);
        }
        if constexpr (NM == 2) {
#pragma unroll
            for (int q = 0; q < 9; q++)
                if (q != 4) {
                    if (o.il == 19 + q) add(19 + q, o.el);
                    if (o.ir == 28 + q) add(28 + q, o.er);
                }
        }
    }
    __syncthreads();
    double *pb = A.pbd[D] + (long)n * S.NG;
    for (int q = threadIdx.x; q < NT; q += 64) {
        const int i = c0[0] + q % TI, j = c0[1] + (q / TI) % TJ, k = c0[2] + q / (TI * TJ);
        if (i <= c1[0] && j <= c1[1] && k <= c1[2]) pb[gidx(B, i, j, k)] = acc[q];
    }
}

template <int NM, bool SMALL>
__global__ __launch_bounds__(64) void k_adj_stencil(DS S, AD A)
{
    __shared__ double acc[ADJ_CELLS[SMALL]];
    const int n0 = S.npv * A.ntiles[0], n1 = n0 + S.npv * A.ntiles[1], w = blockIdx.x;
    if (w < n0) adj_stencil_dir<0, NM, SMALL>(S, A, w, acc);
    else if (w < n1) adj_stencil_dir<1, NM, SMALL>(S, A, w - n0, acc);
    else adj_stencil_dir<2, NM, SMALL>(S, A, w - n1, acc);
}

// Cell sources of one interior cell: the mass transfer, SST, BDF.  MODELS:
// the instantiation with the Kunz / Singhal / Schnerr-Sauer / Lee sources
// (a full EOS of the cell) and the DES length scales, as k_combine<true>.
template <bool MODELS>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_cell_vjp(DS S, AD A)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= S.NC) return;
    const BlkD &B = S.b[find_blk(S, t, 0)];
    const Par &P = S.P;
    const int npv = S.npv;
    int i, j, k;
    cell_of(B, t - B.c0, i, j, k);
    const long g = gidx(B, i, j, k);
    const bool sst = P.iturb == 0;
    double rb[NPV], pc[NPV], d[ND], gr[5][3], f6[6][3], iv = 1.0;
    for (int n = 0; n < NPV; n++) {
        rb[n] = n < npv ? A.rb[(long)n * S.NC + t] : 0.0;
        pc[n] = n < npv ? S.pv[(long)n * S.NG + g] : 0.0;
    }
    for (int m = 0; m < ND; m++) d[m] = S.dc[m * S.NG + g];
    const double vol = S.vol[widx(B, i, j, k)], ydn = sst ? S.ydn[widx(B, i, j, k)] : 1.0;
    const double mut = S.mut ? S.mut[g] : 0.0;
    if (sst) {
        cell_faces(S, B, i, j, k, f6);
        iv = 1.0 / vol;
        const long sy = B.nx, sz = (long)B.nx * B.ny;
        for (int v = 0; v < 5; v++) {
            const int n = v < 3 ? v + 1 : v + 4;
            const double *x = S.pv + (long)n * S.NG + g;
            double x7[7][NPV];
            x7[0][0] = x[-1]; x7[1][0] = x[0]; x7[2][0] = x[1];
            x7[3][0] = x[-sy]; x7[4][0] = x[sy]; x7[5][0] = x[-sz]; x7[6][0] = x[sz];
            gg_grad<double>(x7, 0, f6, iv, gr[v]);
        }
    } else {
        for (int v = 0; v < 5; v++) for (int c = 0; c < 3; c++) gr[v][c] = 0.0;
        for (int q = 0; q < 6; q++) for (int c = 0; c < 3; c++) f6[q][c] = 0.0;
    }
    SourceBar o;
    source_back<MODELS>(P, pc, d, gr, f6, vol, ydn, mut, rb, o);
    if (A.dmut && sst) {
        // the cell's eddy-viscosity bar: its sources' share and its six
        // viscous faces' (the left cell of its + faces, the right cell of
        // its - faces), the eddy viscosity being a state function
        double mb = o.mut;
        for (int D = 0; D < 3; D++) {
            mb += A.mtb[D][fidx(B, D, i, j, k)];
            mb += A.mtb[D][S.NF[D] + fidx(B, D, i - (D == 0), j - (D == 1), k - (D == 2))];
        }
        if (mb != 0.0) eddy_back(mb, pc, d, gr, ydn, o);
    }
    for (int n = 0; n < NPV; n++) if (n < npv) A.cb[(long)n * S.NC + t] = o.pc[n];
    if (sst)
        for (int v = 0; v < 5; v++)
            for (int c = 0; c < 3; c++) A.cb[(long)(npv + 3 * v + c) * S.NC + t] = 0.5 * iv * o.g[v][c];
    A.cdb[t] = o.rho;
    A.cdb[S.NC + t] = o.h;
    A.cdb[2 * S.NC + t] = o.mu;
    for (int q = 0; q < 3; q++) A.csb[(long)q * S.NC + t] = o.sc[q];
}

// The rest of pv_bar of every ghosted cell, added to what k_adj_stencil left:
// the bars of its neighbours' sources, and its property bars (from the faces
// whose cell it is and from its own sources) taken through its EOS, in a
// fixed order.
// Registers: the EOS terms take all 512 of one wavefront a SIMD; held to 256 it
// kept 1.1 KB a lane in scratch memory (128x64x64: 634 us, now 345).
__global__ __launch_bounds__(128) void k_adj_cells(DS S, AD A)
{
    long gl = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (gl >= S.NG) return;
    const BlkD &B = S.b[find_blk(S, gl, 1)];
    const Par &P = S.P;
    const int npv = S.npv;
    const long r = gl - B.g0;
    const int i = (int)(r % B.nx) - 1, j = (int)((r / B.nx) % B.ny) - 1, k = (int)(r / ((long)B.nx * B.ny)) - 1;
    const bool visc = P.iturb >= -2, turb = P.iturb == 0, first = P.nmuscl == 0, sensor = P.nscheme == 2 || P.nscheme == 3;
    double rho = 0.0, h = 0.0, c2 = 0.0, ht = 0.0, mu = 0.0, kap = 0.0;
    for (int D = 0; D < 3; D++) {
        const long NF = S.NF[D];
        for (int sd = 0; sd < 2; sd++) {       // the face whose left (right) cell this is
            const int fi = i - (sd && D == 0), fj = j - (sd && D == 1), fk = k - (sd && D == 2);
            if (!face_exists(B, D, fi, fj, fk)) continue;
            const long f = fidx(B, D, fi, fj, fk);
            if (first) {
                rho += A.fp[D][(long)(3 * sd) * NF + f];
                h += A.fp[D][(long)(3 * sd + 1) * NF + f];
                if (sensor) c2 += A.fp[D][(long)(3 * sd + 2) * NF + f];
            }
            if (visc) {
                mu += A.vp[D][f];
                kap += A.vp[D][NF + f];
                if (turb) {
                    rho += A.vp[D][2 * NF + f];
                    ht += A.vp[D][(3 + sd) * NF + f];
                }
            }
        }
    }
    double acc[NPV];
    for (int n = 0; n < NPV; n++) acc[n] = 0.0;
    const bool inside = interior_cell(B, i, j, k);
    if (inside) {
        const long ct = cidx(B, i, j, k);
        for (int n = 0; n < NPV; n++) if (n < npv) acc[n] = A.cb[(long)n * S.NC + ct];
        rho += A.cdb[ct];
        h += A.cdb[S.NC + ct];
        mu += A.cdb[2 * S.NC + ct];
    }
    if (turb) {
        // the Green-Gauss gradients' transpose: a cell's gradient of x is
        // the sum over its faces of the outward face vector times the mean
        // of x on the two sides, over its volume (A.cb holds half the bar
        // over the volume), so this cell's value meets the cell across each
        // of its faces there, and its own gradient at all six
        double own[3] = {0.0, 0.0, 0.0};
        for (int q = 0; q < 6; q++) {
            const int D = q >> 1, hi = q & 1, e = hi ? 1 : -1;
            const int si = i + (D == 0 ? e : 0), sj = j + (D == 1 ? e : 0), sk = k + (D == 2 ? e : 0);
            const bool nb = interior_cell(B, si, sj, sk);
            if (!inside && !nb) continue;
            double f[3];
            face_vec(S, B, D, hi ? i : si, hi ? j : sj, hi ? k : sk, f);
            for (int c = 0; c < 3; c++) own[c] += hi ? f[c] : -f[c];
            if (!nb) continue;
            const double *gb = A.cb + (long)npv * S.NC + cidx(B, si, sj, sk);
            for (int v = 0; v < 5; v++) {
                const double w = f[0] * gb[(3L * v) * S.NC] + f[1] * gb[(3L * v + 1) * S.NC] + f[2] * gb[(3L * v + 2) * S.NC];
                acc[v < 3 ? v + 1 : v + 4] += hi ? -w : w;
            }
        }
        if (inside) {
            const double *gb = A.cb + (long)npv * S.NC + cidx(B, i, j, k);
            for (int v = 0; v < 5; v++)
                acc[v < 3 ? v + 1 : v + 4] += own[0] * gb[(3L * v) * S.NC] + own[1] * gb[(3L * v + 1) * S.NC] + own[2] * gb[(3L * v + 2) * S.NC];
        }
    }
    if (rho != 0.0 || h != 0.0 || c2 != 0.0 || ht != 0.0 || mu != 0.0 || kap != 0.0) {
        double dcb[ND], gx[4];
        for (int m = 0; m < ND; m++) dcb[m] = 0.0;
        dcb[D_RHO] = rho; dcb[D_H] = h; dcb[D_C2] = c2; dcb[D_HT] = ht; dcb[D_MU] = mu; dcb[D_KAP] = kap;
        const double x4[4] = {S.pv[gl] + P.pref, S.pv[4 * S.NG + gl], S.pv[5 * S.NG + gl], S.pv[6 * S.NG + gl]};
        eos_adj(P.iturb != -3, x4, dcb, gx);
        acc[0] += gx[0]; acc[4] += gx[1]; acc[5] += gx[2]; acc[6] += gx[3];
    }
    for (int n = 0; n < NPV; n++) if (n < npv) {
        const long q = (long)n * S.NG + gl;
        A.pb[q] = ((A.pbd[0][q] + A.pbd[1][q]) + A.pbd[2][q]) + acc[n];
    }
}

// deterministic sum of n doubles in two stages: workgroup b sums its strided
// share (q = b*256 + t + k*256*gridDim) by a fixed tree into part[b]; then
// one workgroup sums the parts the same way.  The order never depends on
// timing, so the result is reproducible bit for bit.
constexpr int SUM_WG = 512;
__global__ __launch_bounds__(256) void k_sum_fixed(const double *a, long n, double *part)
{
    __shared__ double sh[256];
    double s = 0.0;
    for (long q = (long)blockIdx.x * 256 + threadIdx.x; q < n; q += 256L * gridDim.x) s += a[q];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// deterministic sum over q of w[q] * (a[q] - b[q]) * inv_h2, strided as k_sum_fixed
__global__ __launch_bounds__(256) void k_dotdiff_fixed(const double *w, const double *a, const double *b, long n,
                                                       double inv_h2, double *part)
{
    __shared__ double sh[256];
    double s = 0.0;
    for (long q = (long)blockIdx.x * 256 + threadIdx.x; q < n; q += 256L * gridDim.x) s += w[q] * ((a[q] - b[q]) * inv_h2);
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int v = 128; v > 0; v >>= 1) {
        if ((int)threadIdx.x < v) sh[threadIdx.x] += sh[threadIdx.x + v];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// The stencil pass takes the small tiles below this many large ones (times the
// variables): two rounds of the wavefronts that fit the chip (two a SIMD).
// 64x32x32 cells, 7 variables, TVD: 1575 large tiles take 161 us, the small
// ones 113; 53x41x27, 9 variables, MLP: 1728, 396 and 358; 128x64x64, 9
// variables, MLP: 10935, 1577 and 1712.
constexpr long ADJ_FEW = 4096;

int adj_alloc(cav3d_ctx *c)
{
    if (c->adj_ready) return 0;
    DS &S = c->S;
    const int npv = c->npv;
    const bool visc = S.P.iturb >= -2, turb = S.P.iturb == 0;
    int rc;
    if ((rc = dalloc(c, &c->a_rb, (long)npv * S.NC)) || (rc = dalloc(c, &c->a_cb, (long)(npv + (turb ? 15 : 0)) * S.NC)) ||
        (rc = dalloc(c, &c->a_cdb, 3L * S.NC)) || (rc = dalloc(c, &c->a_csb, 3L * S.NC)) || (rc = dalloc(c, &c->a_pb, (long)npv * S.NG)) || (rc = dalloc(c, &c->a_pbd, 3L * npv * S.NG)) ||
        (rc = dalloc(c, &c->a_sum, 16 + 16L * SUM_WG)))
        return rc;
    for (int d = 0; d < 3; d++)
        if ((rc = dalloc(c, &c->a_w[d], 2L * npv * S.NF[d])) || (rc = dalloc(c, &c->a_cell[d], S.NF[d])) ||
            (rc = dalloc(c, &c->a_fp[d], S.P.nmuscl == 0 ? 6L * S.NF[d] : 1L)) ||
            (rc = dalloc(c, &c->a_vb[d], visc ? (turb ? 23L : 15L) * S.NF[d] : 1L)) ||
            (rc = dalloc(c, &c->a_vp[d], visc ? 5L * S.NF[d] : 1L)) ||
            (rc = dalloc(c, &c->a_snb[d], (S.P.nscheme == 2 || S.P.nscheme == 3) ? 18L * S.NF[d] : 1L)) ||
            (rc = dalloc(c, &c->a_ub[d], S.NF[d])) || (rc = dalloc(c, &c->a_mtb[d], turb ? 2L * S.NF[d] : 1L)))
            return rc;
    // tiles of the stencil pass over every block's ghosted cells
    std::vector<int> tl;
    int first[3];
    for (c->a_small = 0;; c->a_small++) {
        tl.clear();
        for (int d = 0; d < 3; d++) {
            const int *t = ADJ_TILE[c->a_small][d];
            first[d] = (int)tl.size();
            for (int b = 0; b < c->nb; b++) {
                const BlkD &B = c->blk[b];
                for (int k = -1; k <= B.K + 3; k += t[2])
                    for (int j = -1; j <= B.J + 3; j += t[1])
                        for (int i = -1; i <= B.I + 3; i += t[0]) {
                            const int t4[4] = {b, i, j, k};
                            tl.insert(tl.end(), t4, t4 + 4);
                        }
            }
            c->a_ntiles[d] = (int)(tl.size() - first[d]) / 4;
        }
        if (c->a_small || npv * (long)tl.size() / 4 >= ADJ_FEW) break;
    }
    if ((rc = dalloc(c, &c->a_tiles[0], tl.size()))) return rc;
    for (int d = 1; d < 3; d++) c->a_tiles[d] = c->a_tiles[0] + first[d];
    HIPCHK(hipMemcpyAsync(c->a_tiles[0], tl.data(), tl.size() * sizeof(int), hipMemcpyHostToDevice, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    c->adj_ready = true;
    return 0;
}

int launch_vjp(cav3d_ctx *c, int dmut = 0)
{
    DS &S = c->S;
    AD A;
    A.rb = c->a_rb;
    A.dmut = dmut;
    for (int d = 0; d < 3; d++) {
        A.w[d] = c->a_w[d]; A.cell[d] = c->a_cell[d]; A.snb[d] = c->a_snb[d]; A.fp[d] = c->a_fp[d];
        A.vb[d] = c->a_vb[d]; A.vp[d] = c->a_vp[d]; A.ub[d] = c->a_ub[d]; A.mtb[d] = c->a_mtb[d];
    }
    A.cb = c->a_cb; A.cdb = c->a_cdb; A.csb = c->a_csb; A.pb = c->a_pb;
    for (int d = 0; d < 3; d++) { A.tiles[d] = c->a_tiles[d]; A.ntiles[d] = c->a_ntiles[d]; A.pbd[d] = c->a_pbd + (long)d * S.npv * S.NG; }
    const bool sensor = S.P.nscheme == 2 || S.P.nscheme == 3;
    const int npv = S.npv;
    FluxWgs g;
    for (int d = 0; d < 3; d++) g.n[d] = nblk(S.NF[d], 128);
    const dim3 fg((g.n[0] + g.n[1] + g.n[2]) * (S.P.iturb >= -2 ? 2 : 1));
    if (sensor) hipLaunchKernelGGL(k_faces_vjp<true>, fg, dim3(128), 0, c->st, S, A, g);
    else hipLaunchKernelGGL(k_faces_vjp<false>, fg, dim3(128), 0, c->st, S, A, g);
    // the stencil pass and the cell sources run beside each other and are
    // joined before the cells' pass
    hipEventRecord(c->fork, c->st);
    hipStreamWaitEvent(c->side, c->fork, 0);
    if (S.P.ides > 0 || S.P.ncav >= 2) hipLaunchKernelGGL(k_cell_vjp<true>, dim3(nblk(S.NC, 128)), dim3(128), 0, c->side, S, A);
    else hipLaunchKernelGGL(k_cell_vjp<false>, dim3(nblk(S.NC, 128)), dim3(128), 0, c->side, S, A);
    const dim3 tg((unsigned)(npv * (c->a_ntiles[0] + c->a_ntiles[1] + c->a_ntiles[2])));
    auto stencil = [&](auto small) {
        constexpr bool SMALL = decltype(small)::value;
        if (S.P.nmuscl == 0) hipLaunchKernelGGL((k_adj_stencil<0, SMALL>), tg, dim3(64), 0, c->st, S, A);
        else if (S.P.nmuscl == 1) hipLaunchKernelGGL((k_adj_stencil<1, SMALL>), tg, dim3(64), 0, c->st, S, A);
        else hipLaunchKernelGGL((k_adj_stencil<2, SMALL>), tg, dim3(64), 0, c->st, S, A);
    };
    if (c->a_small) stencil(std::true_type());
    else stencil(std::false_type());
    hipEventRecord(c->join, c->side);
    hipStreamWaitEvent(c->st, c->join, 0);
    hipLaunchKernelGGL(k_adj_cells, dim3(nblk(S.NG, 128)), dim3(128), 0, c->st, S, A);
    return 0;
}

// every block's res_bar (the calrhs res layout, blocks concatenated) into a_rb
int upload_res_bar(cav3d_ctx *c, const double *res_bar)
{
    int rc;
    if ((rc = adj_alloc(c))) return rc;
    DS &S = c->S;
    const int npv = c->npv;
    long maxn = 0;
    for (int b = 0; b < c->nb; b++) maxn = std::max(maxn, (long)npv * c->blk[b].ng);
    if ((rc = ensure_stage(c, maxn))) return rc;
    long off = 0;
    for (int b = 0; b < c->nb; b++) {
        const BlkD &B = c->blk[b];
        HIPCHK(hipMemcpyAsync(c->stage, res_bar + off, (long)npv * B.nc * sizeof(double), hipMemcpyHostToDevice, c->st));
        hipLaunchKernelGGL(k_cell_from_aos, dim3(nblk(B.nc, 256)), dim3(256), 0, c->st, (const double *)c->stage, npv, S.NC,
                           B.c0, c->a_rb, B.nc);
        HIPCHK(hipStreamSynchronize(c->st));
        off += (long)npv * B.nc;
    }
    return 0;
}

// the fixed-order sum of n values at src into a_sum[slot]
void sum_into(cav3d_ctx *c, const double *src, long n, int slot)
{
    double *part = c->a_sum + 16 + (long)SUM_WG * slot;
    hipLaunchKernelGGL(k_sum_fixed, dim3(SUM_WG), dim3(256), 0, c->st, src, n, part);
    hipLaunchKernelGGL(k_sum_fixed, dim3(1), dim3(256), 0, c->st, (const double *)part, (long)SUM_WG, c->a_sum + slot);
}

}  // namespace

extern "C" {

static int rhs_vjp_run(cav3d_ctx *c, const double *res_bar, double *pv_bar, double *scal_bar, int dmut, const char *name)
{
    if (!c || !res_bar || !pv_bar) return fail(std::string("bad argument to ") + name, -1);
    int rc;
    if ((rc = upload_res_bar(c, res_bar))) return rc;
    DS &S = c->S;
    const int npv = c->npv;
    long off = 0;
    if (c->profile) hipEventRecord(c->ev[10], c->st);
    launch_vjp(c, dmut);
    if (c->profile) {
        hipEventRecord(c->ev[11], c->st);
        hipEventSynchronize(c->ev[11]);
        float ms;
        hipEventElapsedTime(&ms, c->ev[10], c->ev[11]);
        c->prof_ms[8] = ms;
    }
    if ((rc = check_launch(name))) return rc;
    if (scal_bar) {
        const double *src[5] = {c->a_pb, c->a_ub[0], c->a_ub[1], c->a_ub[2], c->a_csb};
        const long len[5] = {S.NG, S.NF[0], S.NF[1], S.NF[2], S.NC};
        for (int q = 0; q < 5; q++) sum_into(c, src[q], len[q], q);
    }
    off = 0;
    for (int b = 0; b < c->nb; b++) {
        const BlkD &B = c->blk[b];
        hipLaunchKernelGGL(k_soa_to_aos, dim3(nblk(B.ng, 256)), dim3(256), 0, c->st, (const double *)c->a_pb, npv, S.NG, B.g0,
                           c->stage, B.ng);
        if ((rc = copy_out(c, pv_bar + off, c->stage, (long)npv * B.ng * sizeof(double)))) return rc;
        off += (long)npv * B.ng;
    }
    if (scal_bar) {
        double h[5];
        HIPCHK(hipMemcpyAsync(h, c->a_sum, sizeof(h), hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipStreamSynchronize(c->st));
        scal_bar[0] = h[0];
        scal_bar[1] = ((h[1] + h[2]) + h[3]) + h[4];
    }
    return check_launch(name);
}

int cav3d_rhs_vjp(cav3d_ctx *c, const double *res_bar, double *pv_bar, double *scal_bar)
{
    return rhs_vjp_run(c, res_bar, pv_bar, scal_bar, 0, "cav3d_rhs_vjp");
}

int cav3d_rhs_vjp_eddy(cav3d_ctx *c, const double *res_bar, double *pv_bar, double *scal_bar)
{
    if (c && c->prm.iturb != 0) return fail("cav3d_rhs_vjp_eddy: the eddy viscosity is a state function only under k-omega SST", -1);
    return rhs_vjp_run(c, res_bar, pv_bar, scal_bar, 1, "cav3d_rhs_vjp_eddy");
}

int cav3d_eddy(cav3d_ctx *c)
{
    if (!c) return fail("bad argument to cav3d_eddy", -1);
    if (c->prm.iturb != 0) return fail("cav3d_eddy: the eddy viscosity is computed only under k-omega SST", -1);
    const DS &S = c->S;
    hipLaunchKernelGGL(k_eddy, dim3(nblk(S.NC, 256)), dim3(256), 0, c->st, S);
    return check_launch("cav3d_eddy");
}

int cav3d_rhs_vjp_params(cav3d_ctx *c, const double *res_bar, double *par_bar)
{
    if (!c || !res_bar || !par_bar) return fail("bad argument to cav3d_rhs_vjp_params", -1);
    int rc;
    if ((rc = upload_res_bar(c, res_bar))) return rc;
    DS &S = c->S;
    const int npv = c->npv;
    if (!c->a_save) {
        if ((rc = dalloc(c, &c->a_save, (long)(2 * npv + ND + 1) * S.NG))) return rc;
    }
    launch_vjp(c);
    // the partials at fixed ghost cells
    sum_into(c, c->a_pb, S.NG, 0);
    sum_into(c, c->a_ub[0], S.NF[0], 1);
    sum_into(c, c->a_ub[1], S.NF[1], 2);
    sum_into(c, c->a_ub[2], S.NF[2], 3);
    for (int q = 0; q < 3; q++) sum_into(c, c->a_csb + (long)q * S.NC, S.NC, 4 + q);
    // the boundary fill's share: for a fixed interior every ghost cell is an
    // affine function of the boundary state bc_pv, bc_pressure (the mirror,
    // surface and neighbour cells and the in/out mode do not move), so the
    // product of the ghost-cell bars with its derivative is a central
    // difference of the fill, exact up to rounding.  The characteristic
    // fills also read u_ref (the preconditioned speed of sound at the
    // surface cell), smoothly where the surface cell's normal speed is not
    // u_ref: the eleventh difference.  The fills also read the surface
    // cells' density and speed of sound, which follow p_ref through the EOS:
    // the twelfth difference refills from the interior properties
    // re-evaluated at p_ref +- h.  The fills evaluate the ghost EOS at
    // bc_pv[0] + gauge pressure, so p_ref is exact together with bc_pv[0]
    // when the two are equal (a change of p_ref that moves the boundary
    // state's reference pressure with it).
    double *save_pv = c->a_save, *save_dc = save_pv + (long)npv * S.NG, *save_mut = save_dc + (long)ND * S.NG;
    double *plus = save_mut + S.NG;
    HIPCHK(hipMemcpyAsync(save_pv, S.pv, (long)npv * S.NG * sizeof(double), hipMemcpyDeviceToDevice, c->st));
    HIPCHK(hipMemcpyAsync(save_dc, S.dc, (long)ND * S.NG * sizeof(double), hipMemcpyDeviceToDevice, c->st));
    if (S.mut) HIPCHK(hipMemcpyAsync(save_mut, S.mut, S.NG * sizeof(double), hipMemcpyDeviceToDevice, c->st));
    const Par P0 = S.P;
    double hs[12], share_u = 0.0, share_p = 0.0;
    for (int m = 0; m < 12; m++) {
        double &theta = (m < 9) ? S.P.bc_pv[m] : (m == 9 ? S.P.bc_pressure : (m == 10 ? S.P.uref : S.P.pref));
        const double v0 = theta;
        const double h = v0 != 0.0 ? 1.0e-4 * fabs(v0) : 1.0e-6;
        hs[m] = h;
        theta = v0 + h;
        if (m == 11) hipLaunchKernelGGL(k_eos_cells, dim3(nblk(S.NC, 256)), dim3(256), 0, c->st, S, 1, 0);
        launch_setbc(c);
        HIPCHK(hipMemcpyAsync(plus, S.pv, (long)npv * S.NG * sizeof(double), hipMemcpyDeviceToDevice, c->st));
        theta = v0 - h;
        if (m == 11) hipLaunchKernelGGL(k_eos_cells, dim3(nblk(S.NC, 256)), dim3(256), 0, c->st, S, 1, 0);
        launch_setbc(c);
        theta = v0;
        double *part = c->a_sum + 16 + (long)SUM_WG * (7 + (m % 8));
        hipLaunchKernelGGL(k_dotdiff_fixed, dim3(SUM_WG), dim3(256), 0, c->st, (const double *)c->a_pb, (const double *)plus,
                           (const double *)S.pv, (long)npv * S.NG, 1.0 / (2.0 * h), part);
        hipLaunchKernelGGL(k_sum_fixed, dim3(1), dim3(256), 0, c->st, (const double *)part, (long)SUM_WG, c->a_sum + 7 + m % 8);
        if (m == 7 || m == 11) {
            // a_sum[7..14] hold up to eight results: copy them out before reuse
            double hm[8];
            HIPCHK(hipMemcpyAsync(hm, c->a_sum + 7, sizeof(hm), hipMemcpyDeviceToHost, c->st));
            HIPCHK(hipStreamSynchronize(c->st));
            const int first = m == 7 ? 0 : 8;
            for (int q = first; q <= m; q++) {
                if (q < 10) par_bar[4 + q] = hm[q % 8];
                else if (q == 10) share_u = hm[q % 8];
                else share_p = hm[q % 8];
            }
        }
    }
    S.P = P0;
    HIPCHK(hipMemcpyAsync(S.pv, save_pv, (long)npv * S.NG * sizeof(double), hipMemcpyDeviceToDevice, c->st));
    HIPCHK(hipMemcpyAsync(S.dc, save_dc, (long)ND * S.NG * sizeof(double), hipMemcpyDeviceToDevice, c->st));
    if (S.mut) HIPCHK(hipMemcpyAsync(S.mut, save_mut, S.NG * sizeof(double), hipMemcpyDeviceToDevice, c->st));
    double h[7];
    HIPCHK(hipMemcpyAsync(h, c->a_sum, sizeof(h), hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    par_bar[0] = h[0] + share_p;
    par_bar[1] = (((h[1] + h[2]) + h[3]) + h[4]) + share_u;
    par_bar[2] = h[5];
    par_bar[3] = h[6];
    return check_launch("cav3d_rhs_vjp_params");
}

int cav3d_objective(cav3d_ctx *c, double w_vap, double w_fx, double *J, double *pv_bar, double *dJ_dpref)
{
    if (!c || !J) return fail("bad argument to cav3d_objective", -1);
    DS &S = c->S;
    long nface;
    bool ok;
    std::vector<FSeg> segs = surface_segments(c, nface, ok);
    if (!ok) return fail("cav3d_objective: a surface range is not a block face inside the cells", -2);
    if (nface > 0 && w_fx != 0.0 && !c->xv) return fail("cav3d_objective: the x-force needs the vertex coordinates (cav3d_set_grid)", -1);
    int rc;
    if ((rc = adj_alloc(c))) return rc;
    if (c->a_obj_n < S.NC + nface) {
        if (c->a_obj) { HIPCHK(hipStreamSynchronize(c->st)); HIPCHK(hipFree(c->a_obj)); c->a_obj = nullptr; }
        HIPCHK(hipMalloc((void **)&c->a_obj, 2 * (S.NC + nface) * sizeof(double)));
        c->a_obj_n = S.NC + nface;
    }
    double *val = c->a_obj, *dpr = c->a_obj + c->a_obj_n;
    // pv_bar: zero on the ghost layers, the cells' shares, then each range's faces
    hipLaunchKernelGGL(k_fill, dim3(nblk((long)c->npv * S.NG, 256)), dim3(256), 0, c->st, c->a_pb, 0.0, (long)c->npv * S.NG);
    hipLaunchKernelGGL(k_obj_cells, dim3(nblk(S.NC, POST_WG)), dim3(POST_WG), 0, c->st, S, (const double *)S.vol, w_vap,
                       c->a_pb, val, dpr);
    long off = S.NC;
    if (w_fx != 0.0)
        for (const FSeg &sg : segs) {
            hipLaunchKernelGGL(k_obj_faces, dim3(nblk(sg.n, POST_WG)), dim3(POST_WG), 0, c->st, S, sg, (const double *)c->xv,
                               c->NV, c->v0[sg.b], (const double *)c->xc, w_fx, c->a_pb, val + off, dpr + off);
            off += sg.n;
        }
    sum_into(c, val, off, 0);
    sum_into(c, dpr, off, 1);
    double h[2];
    HIPCHK(hipMemcpyAsync(h, c->a_sum, sizeof(h), hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    *J = h[0];
    if (dJ_dpref) *dJ_dpref = h[1];
    if (pv_bar) {
        const int npv = c->npv;
        long maxn = 0;
        for (int b = 0; b < c->nb; b++) maxn = std::max(maxn, (long)npv * c->blk[b].ng);
        if ((rc = ensure_stage(c, maxn))) return rc;
        long o = 0;
        for (int b = 0; b < c->nb; b++) {
            const BlkD &B = c->blk[b];
            hipLaunchKernelGGL(k_soa_to_aos, dim3(nblk(B.ng, 256)), dim3(256), 0, c->st, (const double *)c->a_pb, npv, S.NG,
                               B.g0, c->stage, B.ng);
            if ((rc = copy_out(c, pv_bar + o, c->stage, (long)npv * B.ng * sizeof(double)))) return rc;
            o += (long)npv * B.ng;
        }
    }
    return check_launch("cav3d_objective");
}

}  // extern "C"

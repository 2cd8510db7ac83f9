// cav3d: the pseudo-time LU-SGS step on MI355X (gfx950).
//
// Layout: every block's ghosted cell arrays (-1:imax+3 etc.) are concatenated
// in one allocation per field and stored structure-of-arrays, i fastest, so a
// wavefront reads 64 consecutive cells of one variable.  Persistent state is
// pv (npv fields) and the eddy viscosity; the 13 cell properties the path
// reads (rho, h, c^2, the eight EOS derivatives, mu, kappa) are kept per cell
// as the reference keeps dv/tv, and are re-derived from pv wherever the
// reference calls the EOS.
//
// One step (t_lusgs%timeinteg, src/update_module.f90:455-733):
//   k_begin               face boundaries; local dt + global min (timestep_module)
//   k_halo / k_bc         interfaces, edges, corners     (bc_module setbc)
//   k_face                reconstruction + EOS + inviscid/viscous face flux of the three directions
//   k_combine             flux differences in the reference's i,j,k order
//                         + Merkle / SST / BDF sources   (rhs_module calrhs)
//   k_lhs_prep            sweep-independent terms of D^-1 and of the Jacobians
//   k_sweep_tile<fwd>     the L (U) sweep: tiles of i-pencils, hyperplane order,
//                         LDS hand-over inside a tile, coherent polls across tiles
//   k_update, k_finish    pv += dq, clip, EOS, norms; SST eddy viscosity
#include "phys.hpp"
#include "copyout.hpp"
#include "sweep_rows.hpp"
#include "../../include/cav3d.h"

#include <hip/hip_runtime.h>
#include <algorithm>
#include <array>
#include <climits>
#include <cstdio>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

using namespace cav;

#define MAXB 16

namespace {

thread_local std::string g_err;
int fail(const std::string &m, int code = -1) { g_err = m; return code; }

#define HIPCHK(x)                                                                    \
    do {                                                                             \
        hipError_t e_ = (x);                                                         \
        if (e_ != hipSuccess) return fail(std::string(#x) + ": " + hipGetErrorString(e_), -3); \
    } while (0)

struct BlkD {
    int I, J, K, nx, ny;
    long g0, c0, w0, f0[3], cx0, ex0, tx0, p0;   // p0: the block's first pencil
    long ng, nc, nw, nf[3], ncx, nex, ntx;
};

struct Seg {          // one boundary range (face BC, edge or corner)
    int b, fn, face, pad;
    int is[3], ie[3], org[3], dir[3], nb[6][3];
    long start;
};

struct Con {          // one interface connection
    int src, dst;
    int is[3], ie[3], isd[3], tm[9];
    long start;
};

struct DS {           // device state, passed by value
    int nb, npv, nbcseg[3], ncon;
    long NG, NC, NW, NF[3], NCX, NEX, NTX, NBC[3], NHALO;
    double *pv, *dc, *mut, *vol, *ydn, *cx, *ex, *tx;
    double *res, *dt, *icav, *itt, *ocut, *rcav, *qq;
    double *img;      // the sweeps' cell records, in pencils with a record of zeros before and after each [NF[0] + 1][RC_N]
    double *xqf, *xqb; // dq of the sweeps [NW][NPV], a cell's values adjacent: forward
                       // the cross-tile values only, backward every cell's
    long NPLANE;      // pencils: sum over blocks of (J-1)(K-1)
    double *ff[3];    // face fluxes [2*npv][NF] (in img's memory)
    double *red;      // norm partials
    double *scal;     // [0] dt min bits, [1] accumulated time, [2..] norms
    Seg *seg[3];
    Con *con;
    BlkD b[MAXB];
    Par P;
};

enum { FN_NONE = 0, FN_WALLINV, FN_WALLVIS, FN_WALLVISKW, FN_INSUB, FN_OUTSUB, FN_FARFIELD, FN_SYM,
       FN_INSUPER, FN_COPY, FN_EMPTY, FN_EDGEWW, FN_EDGEWWKW, FN_EDGENOWALL, FN_CORNERWW,
       FN_CORNERWWKW, FN_CORNERNOWALL };
enum { F_NONE = -1, F_IMIN = 0, F_IMAX, F_JMIN, F_JMAX, F_KMIN, F_KMAX };

// ------------------------------------------------------------ index helpers
__device__ __forceinline__ long gidx(const BlkD &B, int i, int j, int k)
{
    return B.g0 + (long)(i + 1) + (long)B.nx * ((long)(j + 1) + (long)B.ny * (long)(k + 1));
}
__device__ __forceinline__ long cidx(const BlkD &B, int i, int j, int k)
{
    return B.c0 + (long)(i - 2) + (long)(B.I - 1) * ((long)(j - 2) + (long)(B.J - 1) * (long)(k - 2));
}
__device__ __forceinline__ long widx(const BlkD &B, int i, int j, int k)
{
    return B.w0 + (long)(i - 1) + (long)(B.I + 1) * ((long)(j - 1) + (long)(B.J + 1) * (long)(k - 1));
}
// face-vector arrays by axis: 0 -> cx(1:I,1:J+1,1:K+1), 1 -> ex(1:I+1,1:J,1:K+1), 2 -> tx(1:I+1,1:J+1,1:K)
__device__ __forceinline__ void face_vec(const DS &S, const BlkD &B, int ax, int i, int j, int k, double *v)
{
    const double *a;
    long n, o;
    if (ax == 0) { a = S.cx; n = S.NCX; o = B.cx0 + (i - 1) + (long)B.I * ((j - 1) + (long)(B.J + 1) * (k - 1)); }
    else if (ax == 1) { a = S.ex; n = S.NEX; o = B.ex0 + (i - 1) + (long)(B.I + 1) * ((j - 1) + (long)B.J * (k - 1)); }
    else { a = S.tx; n = S.NTX; o = B.tx0 + (i - 1) + (long)(B.I + 1) * ((j - 1) + (long)(B.J + 1) * (k - 1)); }
    v[0] = a[o]; v[1] = a[n + o]; v[2] = a[2 * n + o];
}

__device__ __forceinline__ int find_blk(const DS &S, long t, int which)
{
    int b = 0;
    for (int q = 1; q < S.nb; q++) {
        long o = which == 0 ? S.b[q].c0 : (which == 1 ? S.b[q].g0 : S.b[q].f0[which - 2]);
        if (t >= o) b = q;
    }
    return b;
}

__device__ __forceinline__ void load_cell(const DS &S, const BlkD &B, int i, int j, int k, CellJ &c)
{
    long g = gidx(B, i, j, k);
    for (int n = 0; n < NPV; n++) if (n < S.npv) c.pv[n] = S.pv[n * S.NG + g];
    for (int m = 0; m < ND; m++) c.d[m] = S.dc[m * S.NG + g];
    c.mut = S.mut ? S.mut[g] : 0.0;
    c.vol = S.vol[widx(B, i, j, k)];
}

__device__ __forceinline__ void cell_faces(const DS &S, const BlkD &B, int i, int j, int k, double f6[6][3])
{
    face_vec(S, B, 0, i - 1, j, k, f6[0]);
    face_vec(S, B, 0, i, j, k, f6[1]);
    face_vec(S, B, 1, i, j - 1, k, f6[2]);
    face_vec(S, B, 1, i, j, k, f6[3]);
    face_vec(S, B, 2, i, j, k - 1, f6[4]);
    face_vec(S, B, 2, i, j, k, f6[5]);
}

__device__ __forceinline__ void cell_of(const BlkD &B, long r, int &i, int &j, int &k)
{
    int ni = B.I - 1, nj = B.J - 1;
    i = 2 + (int)(r % ni);
    j = 2 + (int)((r / ni) % nj);
    k = 2 + (int)(r / ((long)ni * nj));
}

// Kernels over faces or cells that read many neighbours keep a workgroup
// inside one block (the blocks' ranges are rounded up to whole workgroups), so
// the block's extents are scalars: a stencil point or a variable is another
// scalar base, and all of a lane's reads share its one 32-bit offset.
// With per-lane 64-bit places and divisions the viscous face kernels took 85
// us a direction at 128x64x64 cells, now 70, the combine 149, now 143, the
// inviscid ones (bound by their arithmetic) 1 % more than now.  (32 bits: a
// block of 2^29 cells would take more than the device's memory.)
constexpr int BLK_WG = 256;
// the workgroup's block, and the lane's item t of that block's n[b] ones
template <class N> __device__ __forceinline__ int wg_block(const DS &S, unsigned w, N n, unsigned &t)
{
    int b = 0;
    for (int q = 0; q + 1 < S.nb; q++) {
        const unsigned m = (unsigned)((n(S.b[q]) + BLK_WG - 1) / BLK_WG);
        if (b == q && w >= m) { w -= m; b = q + 1; }
    }
    t = w * BLK_WG + threadIdx.x;
    return b;
}
// item q (32 bits, the lane's) of a scalar base
template <class T> __device__ __forceinline__ T &at32(T *base, unsigned q)
{
    return *(T *)((char *)base + (size_t)(q * (unsigned)sizeof(T)));
}
template <class T> __device__ __forceinline__ const T &at32(const T *base, unsigned q)
{
    return *(const T *)((const char *)base + (size_t)(q * (unsigned)sizeof(T)));
}
// 32-bit places within block B's arrays: ghosted, cells with one layer around, face vectors of axis AX
__device__ __forceinline__ unsigned gidx32(const BlkD &B, int i, int j, int k)
{
    return (unsigned)(i + 1) + (unsigned)B.nx * ((unsigned)(j + 1) + (unsigned)B.ny * (unsigned)(k + 1));
}
__device__ __forceinline__ unsigned widx32(const BlkD &B, int i, int j, int k)
{
    return (unsigned)(i - 1) + (unsigned)(B.I + 1) * ((unsigned)(j - 1) + (unsigned)(B.J + 1) * (unsigned)(k - 1));
}
template <int AX> __device__ __forceinline__ unsigned vidx32(const BlkD &B, int i, int j, int k)
{
    const unsigned nx = B.I + (AX != 0), ny = B.J + (AX != 1);
    return (unsigned)(i - 1) + nx * ((unsigned)(j - 1) + ny * (unsigned)(k - 1));
}
// face vector of axis AX at place q, di, dj, dk (uniform) further
template <int AX> __device__ __forceinline__ void face_vec32(const DS &S, const BlkD &B, unsigned q, int di, int dj, int dk, double *v)
{
    const long nx = B.I + (AX != 0), ny = B.J + (AX != 1), n = AX == 0 ? S.NCX : AX == 1 ? S.NEX : S.NTX;
    const double *a = (AX == 0 ? S.cx + B.cx0 : AX == 1 ? S.ex + B.ex0 : S.tx + B.tx0) + (di + nx * (dj + ny * dk));
    v[0] = at32(a, q); v[1] = at32(a + n, q); v[2] = at32(a + 2 * n, q);
}

// ------------------------------------------------------------ EOS kernels
// dc (and mut = emutref) of interior cells from pv
__global__ __launch_bounds__(256) void k_eos_cells(DS S, int interior_only, int set_mut)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    long n = interior_only ? S.NC : S.NG;
    if (t >= n) return;
    int b = find_blk(S, t, interior_only ? 0 : 1);
    const BlkD &B = S.b[b];
    long g;
    if (interior_only) {
        int i, j, k;
        cell_of(B, t - B.c0, i, j, k);
        g = gidx(B, i, j, k);
    } else g = t;
    double d[ND];
    mixture_eos<double>(S.pv[g] + S.P.pref, S.pv[4 * S.NG + g], S.pv[5 * S.NG + g], S.pv[6 * S.NG + g], d, S.P.iturb != -3);
    for (int m = 0; m < ND; m++) S.dc[m * S.NG + g] = d[m];
    if (set_mut && S.mut) S.mut[g] = S.P.emutref;
}

// full dv(18), tv(1:2) of every ghosted cell, AoS for the host
__global__ __launch_bounds__(256) void k_eos_full(DS S, long g0, long n, double *dv, double *tv2)
{
    long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    long g = g0 + q;
    double d[ND], full[18];
    mixture_eos<double>(S.pv[g] + S.P.pref, S.pv[4 * S.NG + g], S.pv[5 * S.NG + g], S.pv[6 * S.NG + g], d,
                        S.P.iturb != -3, full);
    for (int m = 0; m < 18; m++) dv[18 * q + m] = full[m];
    tv2[2 * q] = d[D_MU];
    tv2[2 * q + 1] = d[D_KAP];
}

__global__ __launch_bounds__(256) void k_eos_points(Par P, int n, const double *p, const double *t, const double *y1, const double *y2,
                             double *dv, double *tv)
{
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    double d[ND], full[18];
    mixture_eos<double>(p[q], t[q], y1[q], y2[q], d, true, full);
    for (int m = 0; m < 18; m++) dv[18 * q + m] = full[m];
    tv[2 * q] = d[D_MU];
    tv[2 * q + 1] = d[D_KAP];
}

// ------------------------------------------------------------ time step
constexpr unsigned long long DT_NONE = 0x7ff0000000000000ull;   // +inf: scal[0] between two time steps

__device__ __forceinline__ void timestep_cells(const DS &S, unsigned wg)
{
    long t = (long)wg * blockDim.x + threadIdx.x;
    double dt = 1.0e300;
    if (t < S.NC) {
        const BlkD &B = S.b[find_blk(S, t, 0)];
        int i, j, k;
        cell_of(B, t - B.c0, i, j, k);
        CellJ c;
        load_cell(S, B, i, j, k, c);
        double f6[6][3];
        cell_faces(S, B, i, j, k, f6);
        dt = (S.P.local == -1) ? S.P.cfl : local_dt(S.P, c, f6);
        S.dt[t] = dt;
    }
    // wavefront min, workgroup min, then one atomic per workgroup
    // (positive doubles order as their bit patterns)
    __shared__ double wmin[4];
    for (int o = 32; o > 0; o >>= 1) dt = fmin(dt, __shfl_xor(dt, o));
    if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = dt;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = wmin[0];
        for (int q = 1; q < (int)(blockDim.x >> 6); q++) m = fmin(m, wmin[q]);
        if (m < 1.0e299)
            atomicMin(reinterpret_cast<unsigned long long *>(S.scal), (unsigned long long)__double_as_longlong(m));
    }
}

__global__ __launch_bounds__(256) void k_timestep(DS S) { timestep_cells(S, blockIdx.x); }

// the smallest step into the accumulated time, and its place ready for the next time step
__device__ __forceinline__ void time_acc(const DS &S)
{
    unsigned long long *const bits = reinterpret_cast<unsigned long long *>(S.scal);
    double m = __longlong_as_double((long long)bits[0]);
    if (S.P.local == -1) m = S.P.cfl;
    S.scal[1] += m;
    S.scal[2] = m;
    bits[0] = DT_NONE;
}
__global__ __launch_bounds__(64) void k_time_acc(DS S) { if (threadIdx.x == 0 && blockIdx.x == 0) time_acc(S); }

__global__ __launch_bounds__(256) void k_dt_fill(DS S)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < S.NC) S.dt[t] = __longlong_as_double((long long)reinterpret_cast<unsigned long long *>(S.scal)[0]);
}

// ------------------------------------------------------------ boundary conditions
__device__ __forceinline__ void put_cell(const DS &S, long g, const double *pv, const double *d, double mut)
{
    for (int n = 0; n < NPV; n++) if (n < S.npv) S.pv[n * S.NG + g] = pv[n];
    for (int m = 0; m < ND; m++) S.dc[m * S.NG + g] = d[m];
    if (S.mut) S.mut[g] = mut;
}

__device__ void surface_of(const Seg &s, int i, int j, int k, int *o)
{
    o[0] = s.org[0] + s.dir[0] * i;
    o[1] = s.org[1] + s.dir[1] * j;
    o[2] = s.org[2] + s.dir[2] * k;
    switch (s.face) {
    case F_IMIN: o[0] = s.org[0] + s.dir[0] * s.ie[0]; break;
    case F_IMAX: o[0] = s.org[0] + s.dir[0] * s.is[0]; break;
    case F_JMIN: o[1] = s.org[1] + s.dir[1] * s.ie[1]; break;
    case F_JMAX: o[1] = s.org[1] + s.dir[1] * s.is[1]; break;
    case F_KMIN: o[2] = s.org[2] + s.dir[2] * s.ie[2]; break;
    case F_KMAX: o[2] = s.org[2] + s.dir[2] * s.is[2]; break;
    default: break;
    }
}

// outward area vector of a boundary face at its surface cell
__device__ void outward_of(const DS &S, const BlkD &B, int face, const int *s, double *n)
{
    double sg = 1.0;
    switch (face) {
    case F_IMIN: face_vec(S, B, 0, s[0] - 1, s[1], s[2], n); sg = -1.0; break;
    case F_IMAX: face_vec(S, B, 0, s[0], s[1], s[2], n); break;
    case F_JMIN: face_vec(S, B, 1, s[0], s[1] - 1, s[2], n); sg = -1.0; break;
    case F_JMAX: face_vec(S, B, 1, s[0], s[1], s[2], n); break;
    case F_KMIN: face_vec(S, B, 2, s[0], s[1], s[2] - 1, n); sg = -1.0; break;
    default: face_vec(S, B, 2, s[0], s[1], s[2], n); break;
    }
    n[0] *= sg; n[1] *= sg; n[2] *= sg;
}

__device__ void apply_bc_cell(const DS &S, const Seg &s, int i, int j, int k)
{
    const BlkD &B = S.b[s.b];
    const Par &P = S.P;
    const int npv = S.npv;
    const double *rp = P.bc_pv;
    int m[3] = {s.org[0] + s.dir[0] * i, s.org[1] + s.dir[1] * j, s.org[2] + s.dir[2] * k};
    long gm = gidx(B, m[0], m[1], m[2]);
    long gg = gidx(B, i, j, k);
    double pv[NPV], d[ND], mut = 0.0;
    for (int n = 0; n < NPV; n++) if (n < npv) pv[n] = S.pv[n * S.NG + gm];
    for (int q = 0; q < ND; q++) d[q] = S.dc[q * S.NG + gm];
    if (S.mut) mut = S.mut[gm];
    switch (s.fn) {
    case FN_WALLVIS:
        pv[1] = -pv[1]; pv[2] = -pv[2]; pv[3] = -pv[3];
        put_cell(S, gg, pv, d, mut);
        break;
    case FN_WALLVISKW: {
        int o[3];
        surface_of(s, i, j, k, o);
        long gs = gidx(B, o[0], o[1], o[2]);
        double yd = S.ydn[widx(B, o[0], o[1], o[2])];
        double var = 1600.0 * S.dc[D_MU * S.NG + gs] / S.dc[D_RHO * S.NG + gs] / (yd * yd) - pv[8];
        pv[1] = -pv[1]; pv[2] = -pv[2]; pv[3] = -pv[3]; pv[7] = -pv[7]; pv[8] = var;
        put_cell(S, gg, pv, d, -mut);
        break;
    }
    case FN_WALLINV: case FN_SYM: {
        int o[3];
        double n[3];
        surface_of(s, i, j, k, o);
        outward_of(S, B, s.face, o, n);
        n[0] = -n[0]; n[1] = -n[1]; n[2] = -n[2];
        long gs = gidx(B, o[0], o[1], o[2]);
        double ps1 = S.pv[1 * S.NG + gs], ps2 = S.pv[2 * S.NG + gs], ps3 = S.pv[3 * S.NG + gs];
        double dn = ps1 * n[0] + ps2 * n[1] + ps3 * n[2];
        double nn = n[0] * n[0] + n[1] * n[1] + n[2] * n[2];
        double v1 = 2.0 * (ps1 - n[0] * dn / nn) - pv[1];
        double v2 = 2.0 * (ps2 - n[1] * dn / nn) - pv[2];
        double v3 = 2.0 * (ps3 - n[2] * dn / nn) - pv[3];
        pv[1] = v1; pv[2] = v2; pv[3] = v3;
        put_cell(S, gg, pv, d, mut);
        break;
    }
    case FN_INSUB: case FN_OUTSUB: case FN_FARFIELD: case FN_INSUPER: {
        double press = P.bc_pressure;
        if (s.fn == FN_INSUPER) {
            pv[0] = 2.0 * (press - rp[0]) - pv[0];
            for (int q = 1; q < NPV; q++) if (q < npv) pv[q] = 2.0 * rp[q] - pv[q];
            pv[5] = mn(mx(pv[5], 0.0), 1.0);
            pv[6] = mn(mx(pv[6], 0.0), 1.0);
        } else {
            int o[3];
            double n[3], ps[NPV];
            surface_of(s, i, j, k, o);
            outward_of(S, B, s.face, o, n);
            long gs = gidx(B, o[0], o[1], o[2]);
            for (int q = 0; q < NPV; q++) if (q < npv) ps[q] = S.pv[q * S.NG + gs];
            double rs = S.dc[D_RHO * S.NG + gs], cs = S.dc[D_C2 * S.NG + gs];
            double dl = 1.0 / sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
            double vel = (ps[1] * n[0] + ps[2] * n[1] + ps[3] * n[2]) * dl;
            double a = sqrt(sndp2(P, cs, vel * vel));
            int mode = (s.fn == FN_INSUB) ? 0 : 1;
            if (s.fn == FN_FARFIELD) {
                double mach = vel / sqrt(cs);
                if (mach >= 0.0) mode = (mach >= 1.0) ? 2 : 1;
                else mode = (mach <= -1.0) ? 3 : 0;
            }
            if (mode == 0) {
                double var = press - rp[0] + ps[0]
                           - rs * a * (n[0] * (rp[1] - ps[1]) + n[1] * (rp[2] - ps[2]) + n[2] * (rp[3] - ps[3])) * dl;
                pv[0] = var - pv[0];
                pv[1] = 2.0 * (rp[1] + n[0] * 0.5 * var / rs / a * dl) - pv[1];
                pv[2] = 2.0 * (rp[2] + n[1] * 0.5 * var / rs / a * dl) - pv[2];
                pv[3] = 2.0 * (rp[3] + n[2] * 0.5 * var / rs / a * dl) - pv[3];
                for (int q = 4; q < NPV; q++) if (q < npv) pv[q] = 2.0 * rp[q] - pv[q];
                pv[5] = mn(mx(pv[5], 0.0), 1.0);
                pv[6] = mn(mx(pv[6], 0.0), 1.0);
            } else if (mode == 1) {
                double dp = ps[0] + rp[0] - press;
                pv[0] = 2.0 * (press - rp[0]) - pv[0];
                pv[1] = 2.0 * (ps[1] + n[0] * dp / rs / a * dl) - pv[1];
                pv[2] = 2.0 * (ps[2] + n[1] * dp / rs / a * dl) - pv[2];
                pv[3] = 2.0 * (ps[3] + n[2] * dp / rs / a * dl) - pv[3];
            } else if (mode == 3) {
                pv[0] = 2.0 * (press - rp[0]) - pv[0];
                for (int q = 1; q < NPV; q++) if (q < npv) pv[q] = 2.0 * rp[q] - pv[q];
                pv[5] = mn(mx(pv[5], 0.0), 1.0);
                pv[6] = mn(mx(pv[6], 0.0), 1.0);
            }
        }
        double mu_keep[2] = {d[D_MU], d[D_KAP]};
        mixture_eos<double>(pv[0] + rp[0], pv[4], pv[5], pv[6], d, P.iturb != -3);
        if (P.iturb == -3) { d[D_MU] = mu_keep[0]; d[D_KAP] = mu_keep[1]; }
        put_cell(S, gg, pv, d, mut);
        break;
    }
    case FN_COPY:
        put_cell(S, gg, pv, d, mut);
        break;
    case FN_EDGEWW: case FN_EDGEWWKW: case FN_CORNERWW: case FN_CORNERWWKW: {
        const bool corner = (s.fn == FN_CORNERWW || s.fn == FN_CORNERWWKW);
        const int nn = corner ? 6 : 3;
        double pp[NPV];
        for (int q = 0; q < NPV; q++) if (q < npv) pp[q] = -pv[q];
        for (int t = 0; t < nn; t++) {
            const int *nb = s.nb[t];
            if (!corner && nb[0] == 0 && nb[1] == 0 && nb[2] == 0) continue;
            long gn = gidx(B, nb[0] + s.dir[0] * i, nb[1] + s.dir[1] * j, nb[2] + s.dir[2] * k);
            for (int q = 0; q < NPV; q++) if (q < npv) pp[q] = pp[q] - S.pv[q * S.NG + gn];
        }
        pv[1] = pp[1]; pv[2] = pp[2]; pv[3] = pp[3];
        if (s.fn == FN_EDGEWW || s.fn == FN_CORNERWW) {
            if (npv > 7) { pv[7] = pp[7]; pv[8] = pp[8]; }
        } else {
            double yd = S.ydn[widx(B, m[0], m[1], m[2])];
            double var = 800.0 * d[D_MU] / d[D_RHO] / (yd * yd);
            pv[7] = pp[7];
            pv[8] = (corner ? 8.0 : 4.0) * var + pp[8];
        }
        put_cell(S, gg, pv, d, mut);
        break;
    }
    case FN_EDGENOWALL: case FN_CORNERNOWALL: {
        const bool corner = (s.fn == FN_CORNERNOWALL);
        const int nn = corner ? 6 : 3;
        double mt = mut;
        for (int t = 0; t < nn; t++) {
            const int *nb = s.nb[t];
            if (!corner && nb[0] == 0 && nb[1] == 0 && nb[2] == 0) continue;
            long gn = gidx(B, nb[0] + s.dir[0] * i, nb[1] + s.dir[1] * j, nb[2] + s.dir[2] * k);
            for (int q = 0; q < NPV; q++) if (q < npv) pv[q] = pv[q] + S.pv[q * S.NG + gn];
            if (S.mut) mt = mt + S.mut[gn];
        }
        double f = corner ? 1.0 / 7.0 : 1.0 / 3.0;
        for (int q = 0; q < NPV; q++) if (q < npv) pv[q] = f * pv[q];
        mt = f * mt;
        mixture_eos<double>(pv[0] + rp[0], pv[4], pv[5], pv[6], d, P.iturb != -3);
        put_cell(S, gg, pv, d, mt);
        break;
    }
    default: break;
    }
}

__device__ __forceinline__ void bc_cells(const DS &S, int which, unsigned wg)
{
    long t = (long)wg * blockDim.x + threadIdx.x;
    if (t >= S.NBC[which]) return;
    const Seg *sg = S.seg[which];
    int lo = 0, hi = S.nbcseg[which] - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (sg[mid].start <= t) lo = mid; else hi = mid - 1;
    }
    const Seg &s = sg[lo];
    long r = t - s.start;
    int ni = s.ie[0] - s.is[0] + 1, nj = s.ie[1] - s.is[1] + 1;
    int i = s.is[0] + (int)(r % ni);
    int j = s.is[1] + (int)((r / ni) % nj);
    int k = s.is[2] + (int)(r / ((long)ni * nj));
    apply_bc_cell(S, s, i, j, k);
}
// acc: the launch also takes the time step's minimum (it follows k_begin)
__global__ __launch_bounds__(256) void k_bc(DS S, int which, int acc)
{
    if (acc && blockIdx.x == 0 && threadIdx.x == 0) time_acc(S);
    bc_cells(S, which, blockIdx.x);
}

// interface copy: the sending block's cells to the donor block's ghost cells
__global__ __launch_bounds__(256) void k_halo(DS S)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= S.NHALO) return;
    int lo = 0, hi = S.ncon - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (S.con[mid].start <= t) lo = mid; else hi = mid - 1;
    }
    const Con &c = S.con[lo];
    long r = t - c.start;
    int ni = c.ie[0] - c.is[0] + 1, nj = c.ie[1] - c.is[1] + 1;
    int di = (int)(r % ni), dj = (int)((r / ni) % nj), dk = (int)(r / ((long)ni * nj));
    int ii = c.tm[0] * di + c.tm[1] * dj + c.tm[2] * dk + c.isd[0];
    int jj = c.tm[3] * di + c.tm[4] * dj + c.tm[5] * dk + c.isd[1];
    int kk = c.tm[6] * di + c.tm[7] * dj + c.tm[8] * dk + c.isd[2];
    long gs = gidx(S.b[c.src], c.is[0] + di, c.is[1] + dj, c.is[2] + dk);
    long gd = gidx(S.b[c.dst], ii, jj, kk);
    for (int n = 0; n < NPV; n++) if (n < S.npv) S.pv[n * S.NG + gd] = S.pv[n * S.NG + gs];
    for (int m = 0; m < ND; m++) S.dc[m * S.NG + gd] = S.dc[m * S.NG + gs];
    if (S.mut) S.mut[gd] = S.mut[gs];
}

// ------------------------------------------------------------ face fluxes
// Direction D: normal axis D, first transverse axis E=(D+1)%3, second T=(D+2)%3,
// matching the reference's stencil orderings (src/rhs_module.f90:288-312,
// 374-398, 460-484): ll = 1 + dn + 2(de+1) + 6(dt+1) for dn in {0,1}.
// face of direction D handled by thread t: its (i,j,k) (the left cell) and block
template <int D>
__device__ __forceinline__ const BlkD &face_of(const DS &S, long t, int &i, int &j, int &k)
{
    int b = 0;
    for (int q = 1; q < S.nb; q++) if (t >= S.b[q].f0[D]) b = q;
    const BlkD &B = S.b[b];
    long r = t - B.f0[D];
    if (D == 0) { i = 1 + (int)(r % B.I); j = 2 + (int)((r / B.I) % (B.J - 1)); k = 2 + (int)(r / ((long)B.I * (B.J - 1))); }
    else if (D == 1) { i = 2 + (int)(r % (B.I - 1)); j = 1 + (int)((r / (B.I - 1)) % B.J); k = 2 + (int)(r / ((long)(B.I - 1) * B.J)); }
    else { i = 2 + (int)(r % (B.I - 1)); j = 2 + (int)((r / (B.I - 1)) % (B.J - 1)); k = 1 + (int)(r / ((long)(B.I - 1) * (B.J - 1))); }
    return B;
}

// the same with the workgroup inside one block: t is the face's number there
template <int D>
__device__ __forceinline__ void face_at32(const BlkD &B, unsigned t, int &i, int &j, int &k)
{
    const unsigned ni = D == 0 ? B.I : B.I - 1, nj = D == 1 ? B.J : B.J - 1;
    const unsigned row = t / ni, pl = row / nj;
    i = (D == 0 ? 1 : 2) + (int)(t - row * ni);
    j = (D == 1 ? 1 : 2) + (int)(row - pl * nj);
    k = (D == 2 ? 1 : 2) + (int)pl;
}

// offset of stencil point ll (Fortran numbering) from the face's left cell
template <int D>
__device__ __forceinline__ long stencil_off(const BlkD &B, int ll)
{
    const long st[3] = {1, (long)B.nx, (long)B.nx * B.ny};
    const long sN = st[D], sE = st[(D + 1) % 3], sT = st[(D + 2) % 3];
    int q = ll - 1;
    if (q < 18) return (long)(q & 1) * sN + (long)((q >> 1) % 3 - 1) * sE + (long)(q / 6 - 1) * sT;
    if (q < 27) { q -= 18; return -sN + (long)(q % 3 - 1) * sE + (long)(q / 3 - 1) * sT; }
    if (q < 36) { q -= 27; return 2 * sN + (long)(q % 3 - 1) * sE + (long)(q / 3 - 1) * sT; }
    return q == 36 ? -2 * sN : 3 * sN;
}

// Inviscid flux of every face of direction D (src/rhs_module.f90:282-337 and
// the j/k analogues): reconstruction, clamps, face EOS, Roe / AUSM+-up.
// SENSOR: the Roe-M / AUSMPW+ instantiation (18 stencil pressures, face
// sound speeds); the other schemes run the lighter one.  R: the arithmetic
// of reconstruction, face EOS and flux -- double, or float for the mixed
// precision mode (the state is read in FP64 and rounded once; gauge
// pressure keeps the low-Mach pressure differences; the metastable-vapour
// switch compares against the FP64 saturation pressure).
template <int D, bool SENSOR, class R>
__device__ __forceinline__ void face_flux(const DS &S, unsigned wg)
{
    unsigned t;
    const BlkD &B = S.b[wg_block(S, wg, [](const BlkD &b) { return b.nf[D]; }, t)];
    if (t >= (unsigned)B.nf[D]) return;
    int i, j, k;
    face_at32<D>(B, t, i, j, k);
    const Par &P = S.P;
    const int npv = S.npv;
    const unsigned g9 = gidx32(B, i, j, k);
    const long sN = D == 0 ? 1 : (D == 1 ? (long)B.nx : (long)B.nx * B.ny);
    R c9[NPV], c10[NPV], xl[NPV], xr[NPV];
    R g3[6][3];
    const double *f0 = S.pv + B.g0, *d0 = S.dc + B.g0;
    Par Pi = P;
    Pi.iturb = -3;          // no viscous differences here
    face_recon<R>(Pi, npv, [&](int ll, int n) -> R { return R(at32(f0 + ((long)n * S.NG + stencil_off<D>(B, ll)), g9)); },
                  c9, c10, xl, xr, g3);
    double n3d[3];
    face_vec32<D>(S, B, vidx32<D>(B, i, j, k), 0, 0, 0, n3d);
    const R n3[3] = {R(n3d[0]), R(n3d[1]), R(n3d[2])};
    R rh9[3] = {R(at32(d0 + D_RHO * S.NG, g9)), R(at32(d0 + D_H * S.NG, g9)), R(0)};
    R rh10[3] = {R(at32(d0 + (D_RHO * S.NG + sN), g9)), R(at32(d0 + (D_H * S.NG + sN), g9)), R(0)};
    R fx[NPV];
    if constexpr (SENSOR) {
        // the pressure sensor of Roe-M / AUSMPW+: x(1:18,1) of the face stencil
        R sd[18];
        for (int ll = 1; ll <= 18; ll++) sd[ll - 1] = R(at32(f0 + stencil_off<D>(B, ll), g9));
        rh9[2] = R(at32(d0 + D_C2 * S.NG, g9));
        rh10[2] = R(at32(d0 + (D_C2 * S.NG + sN), g9));
        inviscid_face<R, true>(P, npv, n3, c9, c10, xl, xr, rh9, rh10, fx, sd);
    } else {
        inviscid_face<R, false>(P, npv, n3, c9, c10, xl, xr, rh9, rh10, fx);
    }
    double *out = S.ff[D] + B.f0[D];
    const long NF = S.NF[D];
    for (int n = 0; n < NPV; n++) if (n < npv) at32(out + n * NF, t) = double(fx[n]);
}

// Viscous flux of every face of direction D (src/vsflux_module.f90:182-398),
// with the metric averaging of src/rhs_module.f90:340-357.  R as k_face.
template <int D, class R>
__device__ __forceinline__ void visc_face(const DS &S, unsigned wg)
{
    unsigned t;
    const BlkD &B = S.b[wg_block(S, wg, [](const BlkD &b) { return b.nf[D]; }, t)];
    if (t >= (unsigned)B.nf[D]) return;
    int i, j, k;
    face_at32<D>(B, t, i, j, k);
    const Par &P = S.P;
    const int npv = S.npv;
    const unsigned g9 = gidx32(B, i, j, k);
    const long sN = D == 0 ? 1 : (D == 1 ? (long)B.nx : (long)B.nx * B.ny);
    R g3[6][3] = {};
    R c9[NPV], c10[NPV];
#pragma unroll
    for (int n = 0; n < NPV; n++) {
        c9[n] = c10[n] = R(0);
        if (n >= npv) continue;
        const double *f = S.pv + (B.g0 + (long)n * S.NG);
        auto xs = [&](int ll) -> R { return R(at32(f + stencil_off<D>(B, ll), g9)); };
        c9[n] = R(at32(f, g9));
        c10[n] = R(at32(f + sN, g9));
        if ((n >= 1 && n <= 4) || n >= 7) {
            const int q = (n <= 4) ? n - 1 : n - 3;     // u, v, w, T, k, omega
            g3[q][0] = xs(10) - xs(9);
            g3[q][1] = R(0.0625) * (-xs(1) - xs(2) + xs(5) + xs(6) + R(2) * (-xs(7) - xs(8) + xs(11) + xs(12))
                                    - xs(13) - xs(14) + xs(17) + xs(18));
            g3[q][2] = R(0.0625) * (-xs(1) - xs(2) + xs(13) + xs(14) + R(2) * (-xs(3) - xs(4) + xs(15) + xs(16))
                                    - xs(5) - xs(6) + xs(17) + xs(18));
        }
    }
    constexpr int E = (D + 1) % 3, T = (D + 2) % 3;
    constexpr int dp[3] = {D == 0, D == 1, D == 2}, de[3] = {E == 0, E == 1, E == 2}, dt[3] = {T == 0, T == 1, T == 2};
    double n3d[3], e4d[4][3], t4d[4][3];
    face_vec32<D>(S, B, vidx32<D>(B, i, j, k), 0, 0, 0, n3d);
    const unsigned qe = vidx32<E>(B, i, j, k), qt = vidx32<T>(B, i, j, k);
    // e-family: (P,e-1), (P+1,e-1), (P,e), (P+1,e)
    face_vec32<E>(S, B, qe, -de[0], -de[1], -de[2], e4d[0]);
    face_vec32<E>(S, B, qe, dp[0] - de[0], dp[1] - de[1], dp[2] - de[2], e4d[1]);
    face_vec32<E>(S, B, qe, 0, 0, 0, e4d[2]);
    face_vec32<E>(S, B, qe, dp[0], dp[1], dp[2], e4d[3]);
    // t-family: i faces (P,t-1),(P+1,t-1),(P,t),(P+1,t); j and k faces (P,t-1),(P,t),(P+1,t-1),(P+1,t)
    face_vec32<T>(S, B, qt, -dt[0], -dt[1], -dt[2], t4d[0]);
    face_vec32<T>(S, B, qt, dp[0] - dt[0], dp[1] - dt[1], dp[2] - dt[2], t4d[D == 0 ? 1 : 2]);
    face_vec32<T>(S, B, qt, 0, 0, 0, t4d[D == 0 ? 2 : 1]);
    face_vec32<T>(S, B, qt, dp[0], dp[1], dp[2], t4d[3]);
    R n3[3], e4[4][3], t4[4][3];
    for (int q = 0; q < 3; q++) n3[q] = R(n3d[q]);
    for (int a = 0; a < 4; a++)
        for (int q = 0; q < 3; q++) { e4[a][q] = R(e4d[a][q]); t4[a][q] = R(t4d[a][q]); }
    R gl[2], gr[2], dl[ND], dr[ND];
    const unsigned w = widx32(B, i, j, k);
    const long sW = D == 0 ? 1 : (D == 1 ? (long)(B.I + 1) : (long)(B.I + 1) * (B.J + 1));
    const double *vol = S.vol + B.w0;
    gl[0] = R(at32(vol, w)); gr[0] = R(at32(vol + sW, w));
    gl[1] = R(1); gr[1] = R(1);
    if (S.ydn) { gl[1] = R(at32(S.ydn + B.w0, w)); gr[1] = R(at32(S.ydn + (B.w0 + sW), w)); }
    const double *d0 = S.dc + B.g0;
    for (int m = 0; m < ND; m++) { dl[m] = R(at32(d0 + m * S.NG, g9)); dr[m] = R(at32(d0 + (m * S.NG + sN), g9)); }
    R ml = R(0), mr = R(0);
    if (S.mut) { ml = R(at32(S.mut + B.g0, g9)); mr = R(at32(S.mut + (B.g0 + sN), g9)); }
    R cav[5] = {R(0.5) * (c9[1] + c10[1]), R(0.5) * (c9[2] + c10[2]), R(0.5) * (c9[3] + c10[3]), R(0), R(0)};
    if (npv > 7) { cav[3] = R(0.5) * (c9[7] + c10[7]); cav[4] = R(0.5) * (c9[8] + c10[8]); }
    R fv[NPV];
    visc_flux<R>(P, n3, e4, t4, gl, gr, g3, cav, dl, dr, ml, mr, fv);
    double *out = S.ff[D] + B.f0[D];
    const long NF = S.NF[D];
    for (int n = 0; n < NPV; n++) if (n < npv) at32(out + (npv + n) * NF, t) = double(fv[n]);
}

// All fluxes in one launch: the inviscid faces of the three directions, then
// the viscous ones (they write other halves of the face arrays), each
// direction's workgroups filling the tail of the one before.  V32: the viscous
// faces in FP32 where R is not (AUSMPW+ in the mixed mode).  Six launches on three streams did the same, but an event
// between streams costs some 10 us, and an iteration had three forks and
// joins: it took 210 us at 16x8x8 cells and 162 in single launches on one
// stream, 64x32x32 448 and 409, 128x64x64 1695 and 1671; from a million cells
// on the two were equal (the viscous faces run at two wavefronts per SIMD
// here, three in a launch of their own).
struct FluxWgs { unsigned n[3]; };       // workgroups of each direction
template <int V32, bool SENSOR, class R>
__global__ __launch_bounds__(BLK_WG) void k_face(DS S, FluxWgs g)
{
    using RV = std::conditional_t<V32 != 0, float, R>;
    unsigned w = blockIdx.x;
    if (w < g.n[0]) { face_flux<0, SENSOR, R>(S, w); return; }
    w -= g.n[0];
    if (w < g.n[1]) { face_flux<1, SENSOR, R>(S, w); return; }
    w -= g.n[1];
    if (w < g.n[2]) { face_flux<2, SENSOR, R>(S, w); return; }
    w -= g.n[2];
    if (w < g.n[0]) { visc_face<0, RV>(S, w); return; }
    w -= g.n[0];
    if (w < g.n[1]) { visc_face<1, RV>(S, w); return; }
    visc_face<2, RV>(S, w - g.n[1]);
}

__device__ __forceinline__ long fidx(const BlkD &B, int D, int i, int j, int k)
{
    if (D == 0) return B.f0[0] + (i - 1) + (long)B.I * ((j - 2) + (long)(B.J - 1) * (k - 2));
    if (D == 1) return B.f0[1] + (i - 2) + (long)(B.I - 1) * ((j - 1) + (long)B.J * (k - 2));
    return B.f0[2] + (i - 2) + (long)(B.I - 1) * ((j - 2) + (long)(B.J - 1) * (k - 1));
}

// flux differences in the reference's order, then the cell sources
// MODELS: the instantiation with the Kunz / Singhal / Schnerr-Sauer / Lee
// sources (a full EOS per cell) and the DES length scales; Merkle, no
// cavitation and RANS SST run the lighter one.
template <bool MODELS>
__global__ __launch_bounds__(BLK_WG) void k_combine(DS S)
{
    unsigned t;
    const BlkD &B = S.b[wg_block(S, blockIdx.x, [](const BlkD &b) { return b.nc; }, t)];
    if (t >= (unsigned)B.nc) return;
    const Par &P = S.P;
    const int npv = S.npv;
    const bool visc = (P.iturb >= -2);
    const unsigned nI = B.I - 1, nJ = B.J - 1, row = t / nI, pl = row / nJ;
    const int i = 2 + (int)(t - row * nI), j = 2 + (int)(row - pl * nJ), k = 2 + (int)pl;
    double r[NPV];
#pragma unroll
    for (int D = 0; D < 3; D++) {
        // the cell's lower face of direction D, and from it to the upper one
        const unsigned f = (unsigned)(i - 2) + (nI + (D == 0)) * ((unsigned)(j - 2) + (nJ + (D == 1)) * (unsigned)(k - 2));
        const long up = D == 0 ? 1 : D == 1 ? (long)nI : (long)nI * nJ;
        const double *F = S.ff[D] + B.f0[D];
        const long NF = S.NF[D];
        for (int n = 0; n < NPV; n++) if (n < npv) {
            double a = -(at32(F + (n * NF + up), f) - at32(F + n * NF, f));
            r[n] = (D == 0) ? a : r[n] + a;
            if (visc) r[n] = r[n] + (at32(F + ((npv + n) * NF + up), f) - at32(F + (npv + n) * NF, f));
        }
    }
    const unsigned g = gidx32(B, i, j, k), w = widx32(B, i, j, k);
    const double *f0 = S.pv + B.g0;
    const long NC = S.NC, c0 = B.c0;
    double d[ND], pc[NPV];
    for (int m = 0; m < ND; m++) d[m] = at32(S.dc + (B.g0 + m * S.NG), g);
    for (int n = 0; n < NPV; n++) if (n < npv) pc[n] = at32(f0 + n * S.NG, g);
    double vol = at32(S.vol + B.w0, w);
    if (P.ncav) {
        double rc, rv, ic[4];
        if constexpr (MODELS) {
            if (P.ncav >= 2) {
                double dd[ND], full[18];
                mixture_eos<double>(pc[0] + P.pref, pc[4], pc[5], pc[6], dd, false, full);
                cav_model(P, pc, full, vol, rc, rv, ic);
            } else {
                merkle(P, pc, d, vol, rc, rv, ic);
            }
        } else {
            merkle(P, pc, d, vol, rc, rv, ic);
        }
        r[5] = r[5] + rv - rc;
        for (int q = 0; q < 4; q++) at32(S.icav + (c0 + q * NC), t) = ic[q];
        at32(S.rcav + c0, t) = rc;
        at32(S.rcav + (c0 + NC), t) = rv;
    }
    if (P.iturb == 0) {
        double x7[7][NPV], f6[6][3], src[2], it[4], oc;
        const long ny = B.nx, nz = (long)B.nx * B.ny, to[7] = {-1, 0, 1, -ny, ny, -nz, nz};
        for (int q = 0; q < 7; q++)
            for (int n = 0; n < NPV; n++) if (n < npv) x7[q][n] = at32(f0 + (n * S.NG + to[q]), g);
        const unsigned q0 = vidx32<0>(B, i, j, k), q1 = vidx32<1>(B, i, j, k), q2 = vidx32<2>(B, i, j, k);
        face_vec32<0>(S, B, q0, -1, 0, 0, f6[0]);
        face_vec32<0>(S, B, q0, 0, 0, 0, f6[1]);
        face_vec32<1>(S, B, q1, 0, -1, 0, f6[2]);
        face_vec32<1>(S, B, q1, 0, 0, 0, f6[3]);
        face_vec32<2>(S, B, q2, 0, 0, -1, f6[4]);
        face_vec32<2>(S, B, q2, 0, 0, 0, f6[5]);
        sst_source<MODELS>(P, x7, f6, vol, at32(S.ydn + B.w0, w), d, at32(S.mut + B.g0, g), src, it, oc);
        at32(S.ocut + c0, t) = oc;
        r[7] = r[7] + src[0];
        r[8] = r[8] + src[1];
        for (int q = 0; q < 4; q++) at32(S.itt + (c0 + q * NC), t) = it[q];
    }
    if (P.nsteady > 0) {
        double fx[NPV];
        fx[0] = d[D_RHO];
        fx[1] = d[D_RHO] * pc[1];
        fx[2] = d[D_RHO] * pc[2];
        fx[3] = d[D_RHO] * pc[3];
        fx[4] = d[D_RHO] * (d[D_H] + 0.5 * (pc[1] * pc[1] + pc[2] * pc[2] + pc[3] * pc[3])) - (pc[0] + P.pref);
        for (int n = 5; n < NPV; n++) if (n < npv) fx[n] = d[D_RHO] * pc[n];
        for (int n = 0; n < NPV; n++) if (n < npv) {
            double q1 = at32(S.qq + (c0 + (long)n * NC), t), q2 = at32(S.qq + (c0 + (long)(npv + n) * NC), t);
            double v = (double)P.nsteady * (P.bdf_b * fx[n] - q1) + 0.5 * ((double)P.nsteady - 1.0) * q2;
            r[n] = r[n] - v * vol / P.dt_phy;
        }
    }
    for (int n = 0; n < NPV; n++) if (n < npv) at32(S.res + (c0 + n * NC), t) = r[n];
}

// ------------------------------------------------------------ LU-SGS sweeps
// Per-cell terms of the LU-SGS operator that do not depend on the sweep:
// the diagonal-inverse coefficients and the Jacobian's cell and face terms
// (src/lhs_module.f90:346-457, src/jacobian_module.f90:182-403), written as
// the cells' records.  Bound by HBM (736 bytes a cell written, some 450
// read), so a wavefront turns its 64 records around in LDS, 24 numbers a cell
// at a time, and twelve adjacent lanes write 192 bytes of one record.
// The workgroups from wz on write the records of zeros between the pencils,
// which the face fluxes have been written over.
constexpr int ZERO_ROWS = 64;       // pencils of such a workgroup
__global__ __launch_bounds__(128) void k_lhs_prep(DS S, unsigned wz)
{
    constexpr int CH = 24;
    __shared__ double turn[2][64][CH + 1];
    __shared__ double *to[2][64];
    if (blockIdx.x >= wz) {
        const long r0 = (long)(blockIdx.x - wz) * ZERO_ROWS;
        for (int q = threadIdx.x; q < ZERO_ROWS * (RC_N / 2); q += 128) {
            const long r = r0 + q / (RC_N / 2);
            if (r > S.NPLANE) return;
            int b = 0;
            for (int m = 1; m < S.nb; m++) if (r >= S.b[m].p0) b = m;
            const BlkD &B = S.b[b];
            const long slot = B.f0[0] + (r - B.p0) * B.I;      // (the last pencil's end is the slot behind it)
            *(double2 *)(S.img + slot * RC_N + 2 * (q % (RC_N / 2))) = make_double2(0.0, 0.0);
        }
        return;
    }
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const bool on = t < S.NC;
    const long tc = on ? t : S.NC - 1;
    const BlkD &B = S.b[find_blk(S, tc, 0)];
    const Par &P = S.P;
    int i, j, k;
    cell_of(B, tc - B.c0, i, j, k);
    to[wv][lane] = on ? S.img + fidx(B, 0, i, j, k) * RC_N : nullptr;
    CellJ cc;
    load_cell(S, B, i, j, k, cc);
    double f6[6][3];
    cell_faces(S, B, i, j, k, f6);
    double ic[4] = {0, 0, 0, 0}, it[4] = {0, 0, 0, 0};
    if (P.ncav) for (int m = 0; m < 4; m++) ic[m] = S.icav[m * S.NC + tc];
    if (P.iturb == 0) for (int m = 0; m < 4; m++) it[m] = S.itt[m * S.NC + tc];
    double r[RC_N];
    cell_record(P, S.npv, cc, f6, S.dt[tc], ic, it, r);
    for (int n = 0; n < NPV; n++) r[RC_RES + n] = n < S.npv ? S.res[n * S.NC + tc] : 0.0;
#pragma unroll
    for (int c0 = 0; c0 < RC_N; c0 += CH) {
        const int n = RC_N - c0 < CH ? RC_N - c0 : CH, units = n / 2, per = 64 / units;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < n; q++) turn[wv][lane][q] = r[c0 + q];
        __syncthreads();
        const int u = lane % units, m0 = lane / units;
        for (int m = m0; m < 64; m += per) {
            double *o = to[wv][m];
            if (m0 < per && o)
                *(double2 *)(o + c0 + 2 * u) = make_double2(turn[wv][m][2 * u], turn[wv][m][2 * u + 1]);
        }
    }
}

// ---------------------------------------------------------------- LU-SGS sweeps
// The forward (backward) sweep, src/update_module.f90:486-670:
//   dcv = res + A+(i-1) dq(i-1) + A+(j-1) dq(j-1) + A+(k-1) dq(k-1),  dq = D^-1 dcv
//   (dcv - A-(i+1) dq(i+1) - ... backward), ghost dq = 0.
// Work is split into pencils along i: a 16-lane group owns pencil (j,k) and
// walks i in sweep order.  Lane n accumulates row n of each Jacobian product
// in the reference's order, then the rows are exchanged and lane n evaluates
// component n of D^-1.  dq of a neighbour in another workgroup is published
// with a device-coherent store and read with device-coherent loads; an entry
// still holding the "not yet written" bit pattern is polled again.  Every
// poll is bounded: past the limit the kernel records an error and stops
// waiting, so each wavefront finishes.
constexpr unsigned long long DQ_UNSET = 0x7FF4A5A5A5A5A5A5ull;   // a signalling NaN no arithmetic produces
constexpr long POLL_LIMIT = 1L << 19;

__device__ __forceinline__ double ld_dev(const double *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev(double *p, double v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Tiled sweep: a workgroup owns a tile of TJ x TK pencils of one block and
// walks its hyperplanes s = i + j + k in sweep order with one barrier per
// hyperplane.  A pencil's neighbour inside the tile hands over its dq through
// LDS (by the place of s in the ring); a neighbour in another tile
// through a device-coherent exchange array that holds a cell's values side by
// side (one write of 72 bytes, not nine 8-byte writes to nine lines), waited
// for with a bounded poll.
// Everything a cell reads that does not depend on the sweep (its record and
// the Jacobian operands of its j and k neighbours) is moved ahead of use into
// an LDS stage, so a step's critical path is the dq hand-over and the
// arithmetic.
// Tiles wait only on tiles upstream in j and k.  A workgroup takes its tiles
// from a ticket counter over the topological order, so whatever the number
// of workgroups the device has started, every tile upstream of a started one
// has been taken by a running workgroup: the chain always advances, and the
// launch need not be cooperative.  (Cooperative launches left the stream idle
// for 10 us before the forward sweep and 22 us between the two, beside their
// host time: an iteration of 16x8x8 cells took 0.51 ms with them and 0.30 ms
// with tickets, 64x32x32 0.95 and 0.74, 128x64x64 2.73 and 2.57, state
// transfers included.)
constexpr int TJ = 4, TK = 4;
// LDS stage of one hyperplane (doubles): the tile's sixteen pencils, each its
// cell's F (the sweep's side), Q, GX and RES; then the upstream neighbours in
// other tiles of the four j-edge and the four k-edge pencils, each the F of
// its face towards the tile and its Q (those the next hyperplane's cells
// read, so that every neighbour is in the slab of the step before the one
// that uses it).  A ring of SLABS hyperplanes: a step reads its own slab and
// the next one while the ones after are on their way.  The steps are unrolled
// over the ring, so that the places are constants of the LDS reads.
enum { SLAB_E = TJ * TK * SP_N, SLAB_USED = SLAB_E + (TJ + TK) * SE_N, SLAB_LOADS = (SLAB_USED + 127) / 128, SLAB_N = 128 * SLAB_LOADS };
constexpr int SLABS = 5;

// lane Q of the lane's 16-lane row, by one 64-bit DPP move (no LDS traffic)
struct Dpp {
    template <int Q> __device__ __forceinline__ static double lane(double v)
    {
        return __longlong_as_double(__builtin_amdgcn_mov_dpp(__double_as_longlong(v), 0x150 + Q, 0xF, 0xF, false));
    }
};

// Workgroup barrier for LDS hand-over: this wavefront's LDS accesses are
// complete (lgkmcnt), nothing else is waited for, so global loads and the
// stage LDS-DMA stay in flight across it (a release fence on LDS would also
// wait for every LDS-DMA).  The asm clobbers keep the compiler from moving
// memory accesses across it.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// global address space: a pointer read back from LDS would otherwise be
// generic, and generic loads also count against the LDS wait counter
#define GLOBAL __attribute__((address_space(1)))
constexpr int SWEEP_THREADS = 256 + 64 + 64;   // 16 pencil groups of 16 lanes, a poll and a loader wavefront
constexpr int NEDGE = 2 * 4 * NPV;   // cross-tile dq values a tile reads per step: two edges of four pencils
static_assert(TJ == 4 && TK == 4, "the poll wavefront maps an edge of four pencils");

// Division of labour inside a tile's workgroup:
//  - four pencil wavefronts (16 groups of 16 lanes, lane = row) run the
//    hyperplane steps; they read only LDS and store their cells' results
//    themselves, with no load in flight that a store could wait behind;
//  - a poll wavefront reads, with device-coherent loads, the dq of the
//    upstream cells in other tiles during the step before its use and hands
//    it over through LDS (it is the only wavefront that waits on other tiles);
//  - a loader wavefront fills the stage ahead of the pencils, by LDS-DMA
//    (global memory to LDS, 16 bytes a lane, no registers).
// A step's Jacobian coefficients are formed during the step before from its
// stage without branching on the row, so the dependent chain of a step is
// three row products, the exchange of y and D^-1.
template <bool FWD>
__global__ __launch_bounds__(SWEEP_THREADS) void k_sweep_tile(DS S, const int *tiles, int ntiles, int *err, int *ticket)
{
    // dq hand-over, one LDS object (so that the compiler can tell its reads
    // from the stage LDS-DMA), by the place of the step in the ring: what
    // the step after reads, i.e. the step's dq of the sixteen pencils, the
    // dq of the j / k neighbours of the four and four edge pencils in other
    // tiles, and zeros for a neighbour outside the block
    constexpr int HX = TJ * TK * NPV, HZ = HX + (TJ + TK) * NPV, HN = HZ + NPV;
    __shared__ double hand[SLABS * HN];
    __shared__ double stage[SLABS * SLAB_N];
    __shared__ int gave_up, taken;
    const int npv = S.npv;
    const int sg = FWD ? 1 : -1;
    double *const xq = FWD ? S.xqf : S.xqb;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 15, grp = (threadIdx.x >> 4) & 15;
    if (threadIdx.x == 0) gave_up = 0;
    if (threadIdx.x < SLABS * NPV) hand[threadIdx.x / NPV * HN + HZ + threadIdx.x % NPV] = 0.0;
    for (;;) {
        // the barrier that ends a tile keeps this write behind every read of the last ticket
        if (threadIdx.x == 0) taken = atomicAdd(ticket, 1);
        __syncthreads();
        const int tq = __builtin_amdgcn_readfirstlane(taken);
        if (tq >= ntiles) break;
        const int *td = tiles + 4 * (FWD ? tq : ntiles - 1 - tq);
        const BlkD B = S.b[td[0]];           // a copy: the loops read the block's extents from registers
        const int j0 = td[1], k0 = td[2];
        const int jend = min(j0 + TJ - 1, B.J), kend = min(k0 + TK - 1, B.K);
        // the tile's hyperplane range in sweep order
        const int sa = FWD ? 2 + j0 + k0 : B.I + jend + kend;
        const int sb = FWD ? B.I + jend + kend : 2 + j0 + k0;
        // the pencils whose dq the downstream tiles read (j + 1 and k + 1 edges forward)
        auto down_edge = [](int g) {
            return FWD ? (g % TJ == TJ - 1 || g / TJ == TK - 1) : (g % TJ == 0 || g / TJ == 0);
        };
        if (wave == 5) {
            // Loader wavefront.  Slab n holds hyperplane sa + sg n, slabs from
            // -1 (all pencils before their first cell).  A step n reads slabs
            // n and n + 1; during it slab n + SLABS - 1 is issued, into the
            // place of slab n - 1, which the barrier that ended step n - 1
            // freed, and before its end slab n + 2 has landed: of the slabs
            // issued, the last SLABS - 3 may still be on their way.
            // Lane and transfer (16 bytes) to piece of a record: the 37 pieces
            // of a pencil, F then Q, GX and RES; the 12 of an edge neighbour.
            // Before and past a pencil's ends, and everywhere in a pencil
            // outside the block, it is a record of zeros.
            int l = threadIdx.x - 320;
            asm volatile("" : "+v"(l));          // (worked out per tile: kept across tiles, its pieces end up in scratch memory)
            const double *src[SLAB_LOADS];       // the piece of the coming slab
            int at[SLAB_LOADS];                  // its cell is at - 1 past the pencil's first zero record in sweep order
#pragma unroll
            for (int t = 0; t < SLAB_LOADS; t++) {
                const int u = 64 * t + l;
                int jj, kk, jn, kn, q, early;
                if (u < TJ * TK * SP_N / 2) {
                    const int g = u / (SP_N / 2), c = u % (SP_N / 2);
                    jj = jn = j0 + g % TJ;
                    kk = kn = k0 + g / TJ;
                    q = stage_item(FWD, 2 * c);
                    early = 0;
                } else {
                    const int v = u - TJ * TK * SP_N / 2, e = min(v / (SE_N / 2), TJ + TK - 1), c = v % (SE_N / 2);
                    const bool a = e >= TK;      // a k neighbour
                    jj = j0 + (a ? e - TK : FWD ? 0 : TJ - 1);
                    kk = k0 + (!a ? e : FWD ? 0 : TK - 1);
                    jn = a ? jj : jj - sg;
                    kn = a ? kk - sg : kk;
                    q = edge_item(FWD, a ? 2 : 1, 2 * c);
                    early = 1;
                }
                // cells are numbered 0..I in sweep order, the zero records at
                // the pencil's ends included; slab -1 holds cell at - 1 of it
                at[t] = FWD ? sa - sg - jj - kk - 1 + early : B.I + 1 - (sa - sg - jj - kk) + early;
                const bool in = ((unsigned)(jn - 2) < (unsigned)(B.J - 1)) & ((unsigned)(kn - 2) < (unsigned)(B.K - 1));
                at[t] = in ? at[t] : INT_MIN / 2;        // (stays at the end of the block's first pencil)
                const int c0 = min(max(at[t], 0), B.I), row = in ? jn - 2 + (B.J - 1) * (kn - 2) : 0;
                src[t] = S.img + (B.f0[0] + (long)B.I * row + (FWD ? c0 : B.I - c0)) * RC_N + q;
            }
            const unsigned BI = B.I;
            auto issue = [&](int slot) {
#pragma unroll
                for (int t = 0; t < SLAB_LOADS; t++) {
                    __builtin_amdgcn_global_load_lds((const GLOBAL void *)src[t],
                                                     (__attribute__((address_space(3))) void *)&stage[slot * SLAB_N + 128 * t],
                                                     16, 0, 0);
                    // on to the next cell, from the first zero record to the last
                    src[t] += (unsigned)at[t] < BI ? sg * RC_N : 0;
                    at[t]++;
                }
            };
            // SLABS - 3 slabs of SLAB_LOADS transfers may be outstanding
            static_assert(SLAB_LOADS == 11 && SLABS == 5, "the wait below");
            issue(SLABS - 1);
#pragma unroll
            for (int n = 0; n < SLABS - 1; n++) issue(n);
            asm volatile("s_waitcnt vmcnt(22)" ::: "memory");
            __syncthreads();
            __syncthreads();
            int slot = SLABS - 1;
            for (int s = sa;; s += sg) {
                issue(slot);
                slot = slot == SLABS - 1 ? 0 : slot + 1;
                asm volatile("s_waitcnt vmcnt(22)" ::: "memory");
                lds_barrier();
                if (s == sb) break;
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            continue;
        }
        if (wave == 4) {
            // poll wavefront: item q = lane, lane + 64 of the 72 edge values
            // (edge a = q / 36: the j (a = 0) or k (a = 1) neighbours; pencil
            // e = q / 9 % 4 along the edge; row n = q % 9)
            const int l64 = threadIdx.x - 256;
            const double *dummy = xq + widx(B, min(max(sa - j0 - k0, 2), B.I), j0, k0) * NPV;
            // per lane and tile: item t's value of step s is at xq[at + 9 s],
            // read for lo <= s <= hi (the cell is inside the block and its
            // neighbour too), and goes to the hand-over item to
            long at[2];
            int lo[2], hi[2], to[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int q = min(l64 + 64 * t, NEDGE - 1), a = q / (4 * NPV), e = (q / NPV) % 4, n = q % NPV;
                const int g = a == 0 ? e * TJ + (FWD ? 0 : TJ - 1) : (FWD ? 0 : TK - 1) * TJ + e;
                const int jj = j0 + g % TJ, kk = k0 + g / TJ;
                const int jn = a == 0 ? jj - sg : jj, kn = a == 0 ? kk : kk - sg;
                const bool on = l64 + 64 * t < NEDGE && n < npv && jj <= jend && kk <= kend && jn >= 2 && jn <= B.J && kn >= 2 && kn <= B.K;
                at[t] = widx(B, -jj - kk, jn, kn) * NPV + n;
                lo[t] = on ? 2 + jj + kk : 1;
                hi[t] = on ? B.I + jj + kk : 0;
                to[t] = HX + (a * TK + e) * NPV + n;
            }
            bool n0, n1;
            const double *p0, *p1;
            double v0, v1;
            auto issue = [&](int s) {            // loads for step s (unconditional: the count of loads never varies)
                n0 = s >= lo[0] && s <= hi[0];
                n1 = s >= lo[1] && s <= hi[1];
                p0 = n0 ? xq + at[0] + (long)s * NPV : dummy;
                p1 = n1 ? xq + at[1] + (long)s * NPV : dummy;
                v0 = ld_dev(p0);
                v1 = ld_dev(p1);
            };
            auto deliver = [&](int s, int slot) {    // wait (bounded) for step s's values, then hand them over
                auto unset = [](bool nd, double v) { return nd && (unsigned long long)__double_as_longlong(v) == DQ_UNSET; };
                if (__ballot(unset(n0, v0) || unset(n1, v1))) {
                    long polls = 0;
                    do {
                        // another tile's give-up is read now and then, not on every poll
                        if (++polls > POLL_LIMIT ||
                            ((polls & 255) == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
                            gave_up = 1;
                            v0 = v1 = 0.0;
                            break;
                        }
                        if (unset(n0, v0)) v0 = ld_dev(p0);
                        if (unset(n1, v1)) v1 = ld_dev(p1);
                    } while (__ballot(unset(n0, v0) || unset(n1, v1)));
                }
                hand[to[0] + slot * HN] = n0 ? v0 : 0.0;
                if (l64 < NEDGE - 64) hand[to[1] + slot * HN] = n1 ? v1 : 0.0;
            };
            int slot = SLABS - 1;                // the place of the step before the one whose values are read
            issue(sa);
            deliver(sa, slot);
            __syncthreads();
            __syncthreads();
            for (int s = sa;; s += sg) {
                slot = slot == SLABS - 1 ? 0 : slot + 1;
                // the next step's values are read at the start of this step,
                // while the pencils compute, as late as they can be
                if (s != sb) issue(s + sg);
                if (s != sb) deliver(s + sg, slot);
                lds_barrier();
                if (s == sb) break;
            }
            if (gave_up && l64 == 0) atomicOr(err, 1);
            __syncthreads();
            continue;
        }
        // pencil wavefronts
        const int gj = grp % TJ, gk = grp / TJ;
        const bool mine = lane < npv;
        const int ln = lane < NPV ? lane : 0;
        const RowMap rows = row_map(lane, npv);
        const int j = j0 + gj, k = k0 + gk;
        const bool live = (j <= jend && k <= kend);
        const bool edge = down_edge(grp);
        const int BI = B.I;
        const int jm = j - sg, km = k - sg;
        const bool lj = jm >= j0 && jm <= jend, lk = km >= k0 && km <= kend;
        const bool nj = jm >= 2 && jm <= B.J, nk = km >= 2 && km <= B.K;   // neighbour inside the block
        const bool ej = gj == (FWD ? 0 : TJ - 1), ek = gk == (FWD ? 0 : TK - 1);
        // Places of the stage items: this pencil's, and its j and k
        // neighbours' (a pencil of the tile, or an edge neighbour), each in a
        // slab; of the upstream dq in the hand-over object
        const int mp = grp * SP_N;
        const JacAt ai = jac_at(rows, stage + mp, false, 0),
                    aj = jac_at(rows, stage + (ej ? SLAB_E + gk * SE_N : (grp - sg) * SP_N), ej, 1),
                    ak = jac_at(rows, stage + (ek ? SLAB_E + (TK + gj) * SE_N : (grp - sg * TJ) * SP_N), ek, 2);
        auto cell = [&](int slab) { return row_cell(rows, ai, stage + mp, slab, ln); };
        // (indices into the hand-over object, not pointers chosen among
        // several, so the compiler sees these reads cannot touch the stage)
        const int oi = grp * NPV + ln, oj = (lj ? (grp - sg) * NPV : nj ? HX + gk * NPV : HZ) + ln,
                  ok = (lk ? (grp - sg * TJ) * NPV : nk ? HX + (TK + gj) * NPV : HZ) + ln;
        // where this pencil's results go, from the cell of the first hyperplane on
        const int i0 = sa - j - k;
        double *xe = xq + (widx(B, i0, min(j, B.J), min(k, B.K)) * NPV + lane);
        double *yo = S.img + (fidx(B, 0, i0, min(j, B.J), min(k, B.K)) * RC_N + RC_RES + lane);
        if (lane < NPV) hand[(SLABS - 1) * HN + oi] = 0.0;           // the first step's upstream reads zeros
        double ci[8], cj[8], ck[8];                                  // coefficients of the coming step
        RowCell own;                                                 // its cell
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 8; q++) ci[q] = 0.0;
        row_coef<Dpp>(rows, row_jac(aj, (SLABS - 1) * SLAB_N), cj);
        row_coef<Dpp>(rows, row_jac(ak, (SLABS - 1) * SLAB_N), ck);
        own = cell(0);
        __syncthreads();
        int i = i0, left = (sb - sa) * sg;                           // this step's cell, the steps after it
        // step n of the tile, n mod SLABS = C; false after the last one
        auto step = [&](auto C) {
            constexpr int c = C, before = (c + SLABS - 1) % SLABS, after = (c + 1) % SLABS;
            const bool act = live && i >= 2 && i <= BI;
            // dq of the three upstream neighbours: in the tile from the
            // previous hyperplane, from another tile through the poll wavefront
            const double xi = hand[oi + before * HN], xj = hand[oj + before * HN], xk = hand[ok + before * HN];
            // dcv = res + the three upstream products, in the reference's i, j, k order
            double y = own.res;
            row_apply<Dpp>(ci, xi, y);
            row_apply<Dpp>(cj, xj, y);
            row_apply<Dpp>(ck, xk, y);
            // dq = D^-1 dcv
            const double xn = row_dinv<Dpp>(rows, own, y);
            if (lane < NPV) {
                hand[oi + c * HN] = act ? xn : 0.0;
                // the dq that other tiles wait for goes out at once.  Forward,
                // no other dq is read again (the backward sweep starts from
                // dcv); backward, every cell's is the update's input
                if (act && mine) {
                    if (edge) st_dev(xe, xn);
                    if constexpr (FWD) *yo = y;
                    else if (!edge) *xe = xn;
                }
            }
            xe += sg * NPV;
            if constexpr (FWD) yo += RC_N;
            i += sg;
            // coefficients of the next step (independent of dq): this cell's
            // row through its face to the next cell, and the j / k neighbours
            // of the next cell; and the next cell's own terms
            const RowJac nbj = row_jac(aj, c * SLAB_N), nbk = row_jac(ak, c * SLAB_N);
            row_coef<Dpp>(rows, own.j, ci);
            row_coef<Dpp>(rows, nbj, cj);
            row_coef<Dpp>(rows, nbk, ck);
            own = cell(after * SLAB_N);
            // formed before the barrier (while the poll wavefront may still be
            // waiting), not after it on the next step's path
#pragma unroll
            for (int q = 0; q < 8; q++) asm volatile("" : "+v"(ci[q]), "+v"(cj[q]), "+v"(ck[q]));
#pragma unroll
            for (int q = 0; q < 7; q++) asm volatile("" : "+v"(own.g[q]));
            asm volatile("" : "+v"(own.res), "+v"(own.j.v1), "+v"(own.j.a), "+v"(own.j.b), "+v"(own.j.c), "+v"(own.j.lb), "+v"(own.j.v2), "+v"(own.j.p),
                         "+v"(own.a), "+v"(own.co[0]), "+v"(own.co[1]), "+v"(own.co[2]));
            lds_barrier();
            return left-- > 0;
        };
        static_assert(SLABS == 5, "the steps of the ring");
        while (step(std::integral_constant<int, 0>{}) && step(std::integral_constant<int, 1>{}) && step(std::integral_constant<int, 2>{}) &&
               step(std::integral_constant<int, 3>{}) && step(std::integral_constant<int, 4>{})) {
        }
        __syncthreads();
    }
}

// both exchange arrays to "not yet written", both tile tickets to zero
__device__ __forceinline__ void sweep_reset(const DS &S, long n, int *ticket, unsigned wg)
{
    long t = (long)wg * blockDim.x + threadIdx.x;
    if (t < 2) ticket[t] = 0;
    if (t < n) S.xqf[t] = S.xqb[t] = __longlong_as_double((long long)DQ_UNSET);
}
__global__ __launch_bounds__(256) void k_sweep_reset(DS S, long n, int *ticket) { sweep_reset(S, n, ticket, blockIdx.x); }

// The start of an iteration in one launch: the face boundaries, the time step
// and the sweeps' resets, none of which reads what another writes.  All its
// workgroups take the boundary part's registers (one wavefront a SIMD; the
// time step alone runs at five, the resets at eight), so it gains where
// launches count and loses where the cells do: with the three in launches of
// their own, 16x8x8 cells take 2.7 + 5.4 + 8.7 us and two launches more, here
// 13.8; 128x64x64 14 + 34 + 11, here 75; 192x96x64 28 + 69 + 11, here 164.  The
// launches ran beside each other on three streams before, whose joins cost
// what this loses: an iteration of 192x96x64 cells took 3498 us so, 3499 here.
__global__ __launch_bounds__(256) void k_begin(DS S, unsigned nbc, unsigned nts, long nq, int *ticket)
{
    unsigned w = blockIdx.x;
    if (w < nbc) { bc_cells(S, 0, w); return; }
    w -= nbc;
    if (w < nts) { timestep_cells(S, w); return; }
    sweep_reset(S, nq, ticket, w - nts);
}

// ------------------------------------------------------------ update + norms
// Two wavefronts per SIMD: left to itself the compiler gives the cell's EOS
// 268 registers, one wavefront per SIMD, and the loads go unhidden (159 us
// against 99 us with a small spill, 524288 cells).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_update(DS S)
{
    __shared__ double sred[4][NPV + 1];
    __shared__ long sidx[4];
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const Par &P = S.P;
    const int npv = S.npv;
    double dsq[NPV + 1];
    for (int n = 0; n <= NPV; n++) dsq[n] = 0.0;
    double amax = -1.0;
    long aidx = 0x7fffffffffffffffL;
    if (t < S.NC) {
        int bb = find_blk(S, t, 0);
        const BlkD &B = S.b[bb];
        int i, j, k;
        cell_of(B, t - B.c0, i, j, k);
        long g = gidx(B, i, j, k), w = widx(B, i, j, k);
        double p[NPV], old[NPV];
        for (int n = 0; n < NPV; n++) if (n < npv) { old[n] = S.pv[n * S.NG + g]; p[n] = old[n] + S.xqb[w * NPV + n]; }
        p[0] = mx(-P.pref + 1.0e1, p[0]);
        p[5] = mn(1.0, mx(0.0, p[5]));
        p[6] = mn(1.0, mx(0.0, p[6]));
        if (P.iturb == 0) {
            p[7] = mx(p[7], 1.0e-16);
            p[8] = mx(mx(p[8], 1.0e-16), S.ocut[t]);
        }
        for (int n = 0; n < NPV; n++) if (n < npv) S.pv[n * S.NG + g] = p[n];
        double d[ND];
        mixture_eos<double>(p[0] + P.pref, p[4], p[5], p[6], d, P.iturb != -3);
        for (int m = 0; m < ND; m++) S.dc[m * S.NG + g] = d[m];
        for (int n = 0; n < NPV; n++) if (n < npv) { double q = fabs(old[n] - p[n]); dsq[n] = q * q; }
        double q0 = fabs(old[0] - p[0]);
        if (q0 > 1.0e-12) {
            amax = q0;
            // linear order of the reference's scan: block, then k, j, i
            aidx = ((long)bb << 48) | ((long)k << 32) | ((long)j << 16) | (long)i;
        }
    }
    // wavefront reduction
    for (int o = 32; o > 0; o >>= 1) {
        for (int n = 0; n < NPV; n++) if (n < npv) dsq[n] += __shfl_xor(dsq[n], o);
        double om = __shfl_xor(amax, o);
        long oi = __shfl_xor(aidx, o);
        if (om > amax || (om == amax && oi < aidx)) { amax = om; aidx = oi; }
    }
    int wv = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        for (int n = 0; n < NPV; n++) if (n < npv) sred[wv][n] = dsq[n];
        sred[wv][NPV] = amax;
        sidx[wv] = aidx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double acc[NPV + 1];
        double bm = sred[0][NPV];
        long bi = sidx[0];
        for (int n = 0; n < NPV; n++) if (n < npv) acc[n] = sred[0][n];
        for (int q = 1; q < (int)(blockDim.x >> 6); q++) {
            for (int n = 0; n < NPV; n++) if (n < npv) acc[n] += sred[q][n];
            if (sred[q][NPV] > bm || (sred[q][NPV] == bm && sidx[q] < bi)) { bm = sred[q][NPV]; bi = sidx[q]; }
        }
        double *o = S.red + (long)blockIdx.x * (NPV + 2);
        for (int n = 0; n < NPV; n++) if (n < npv) o[n] = acc[n];
        o[NPV] = bm;
        reinterpret_cast<long *>(o)[NPV + 1] = bi;
    }
}

// fixed-order final reduction of the per-workgroup partials (deterministic)
__device__ __forceinline__ void norm_final(const DS &S, int nwg)
{
    __shared__ double part[256][NPV];
    __shared__ double pm[256];
    __shared__ long pi[256];
    int tid = threadIdx.x;
    double acc[NPV];
    for (int n = 0; n < NPV; n++) acc[n] = 0.0;
    double bm = -1.0;
    long bi = 0x7fffffffffffffffL;
    for (int q = tid; q < nwg; q += 256) {
        const double *o = S.red + (long)q * (NPV + 2);
        for (int n = 0; n < NPV; n++) if (n < S.npv) acc[n] += o[n];
        long oi = reinterpret_cast<const long *>(o)[NPV + 1];
        if (o[NPV] > bm || (o[NPV] == bm && oi < bi)) { bm = o[NPV]; bi = oi; }
    }
    for (int n = 0; n < NPV; n++) part[tid][n] = acc[n];
    pm[tid] = bm;
    pi[tid] = bi;
    __syncthreads();
    // pairwise tree in a fixed pairing: the same inputs always give the same bits
    for (int h = 128; h > 0; h >>= 1) {
        if (tid < h) {
            for (int n = 0; n < NPV; n++) part[tid][n] += part[tid + h][n];
            if (pm[tid + h] > pm[tid] || (pm[tid + h] == pm[tid] && pi[tid + h] < pi[tid])) {
                pm[tid] = pm[tid + h];
                pi[tid] = pi[tid + h];
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        for (int n = 0; n < NPV; n++) if (n < S.npv) S.scal[4 + n] = sqrt(part[0][n]);
        S.scal[4 + NPV] = pm[0];
        reinterpret_cast<long *>(S.scal)[5 + NPV] = pi[0];
    }
}

__device__ __forceinline__ void eddy_cells(const DS &S, unsigned wg)
{
    long t = (long)wg * blockDim.x + threadIdx.x;
    if (t >= S.NC) return;
    const BlkD &B = S.b[find_blk(S, t, 0)];
    int i, j, k;
    cell_of(B, t - B.c0, i, j, k);
    double x7[7][NPV], f6[6][3], d[ND];
    const int di[7] = {-1, 0, 1, 0, 0, 0, 0}, dj[7] = {0, 0, 0, -1, 1, 0, 0}, dk[7] = {0, 0, 0, 0, 0, -1, 1};
    for (int q = 0; q < 7; q++) {
        long gn = gidx(B, i + di[q], j + dj[q], k + dk[q]);
        for (int n = 0; n < NPV; n++) if (n < S.npv) x7[q][n] = S.pv[n * S.NG + gn];
    }
    long g = gidx(B, i, j, k);
    for (int m = 0; m < ND; m++) d[m] = S.dc[m * S.NG + g];
    cell_faces(S, B, i, j, k, f6);
    long w = widx(B, i, j, k);
    S.mut[g] = sst_eddy(x7, f6, S.vol[w], S.ydn[w], d);
}
__global__ __launch_bounds__(256) void k_eddy(DS S) { eddy_cells(S, blockIdx.x); }

// The end of an iteration: the norms' final reduction in the first workgroup,
// the eddy viscosity in the others
__global__ __launch_bounds__(256) void k_finish(DS S, int nwg)
{
    if (blockIdx.x == 0) norm_final(S, nwg);
    else eddy_cells(S, blockIdx.x - 1);
}

// dual time: qq(2) = qq(1), qq(1) = Q(pv, dv)
__global__ __launch_bounds__(256) void k_unsteady_shift(DS S)
{
    long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= S.NC) return;
    const BlkD &B = S.b[find_blk(S, t, 0)];
    int i, j, k;
    cell_of(B, t - B.c0, i, j, k);
    long g = gidx(B, i, j, k);
    const int npv = S.npv;
    double pc[NPV];
    for (int n = 0; n < NPV; n++) if (n < npv) pc[n] = S.pv[n * S.NG + g];
    double rho = S.dc[D_RHO * S.NG + g], h = S.dc[D_H * S.NG + g];
    for (int n = 0; n < NPV; n++) if (n < npv) S.qq[(long)(npv + n) * S.NC + t] = S.qq[(long)n * S.NC + t];
    double q[NPV];
    q[0] = rho;
    q[1] = rho * pc[1];
    q[2] = rho * pc[2];
    q[3] = rho * pc[3];
    q[4] = rho * (h + 0.5 * (pc[1] * pc[1] + pc[2] * pc[2] + pc[3] * pc[3])) - pc[0] - S.P.pref;
    for (int n = 5; n < NPV; n++) if (n < npv) q[n] = rho * pc[n];
    for (int n = 0; n < NPV; n++) if (n < npv) S.qq[(long)n * S.NC + t] = q[n];
}

// ------------------------------------------------------------ layout transposes
// host AoS (m components fastest) <-> device SoA for one block's ghosted cells
__global__ __launch_bounds__(256) void k_aos_to_soa(const double *src, int m, int msrc, int moff, double *dst, long nstride, long g0, long n)
{
    long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    for (int q = 0; q < m; q++) dst[q * nstride + g0 + g] = src[g * msrc + moff + q];
}
__global__ __launch_bounds__(256) void k_soa_to_aos(const double *src, int m, long nstride, long g0, double *dst, long n)
{
    long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    for (int q = 0; q < m; q++) dst[g * m + q] = src[q * nstride + g0 + g];
}
// dv(18) AoS -> compact dc, tv(ntv) AoS -> mu, kappa, mut
__global__ __launch_bounds__(256) void k_dv_to_dc(const double *dv, const double *tv, int ntv, double *dc, double *mut, long nstride, long g0, long n)
{
    long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n) return;
    const int map[11] = {0, 1, 5, 6, 7, 8, 9, 10, 11, 12, 13};
    for (int q = 0; q < 11; q++) dc[q * nstride + g0 + g] = dv[18 * g + map[q]];
    if (ntv >= 2) {
        dc[D_MU * nstride + g0 + g] = tv[ntv * g];
        dc[D_KAP * nstride + g0 + g] = tv[ntv * g + 1];
    }
    if (ntv == 3 && mut) mut[g0 + g] = tv[ntv * g + 2];
}
// interior-cell arrays (c-indexed SoA, m components) -> reference AoS (m,2:imax,...)
__global__ __launch_bounds__(256) void k_cell_to_aos(const double *src, int m, long nstride, long c0, double *dst, long n)
{
    long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    for (int a = 0; a < m; a++) dst[q * m + a] = src[a * nstride + c0 + q];
}
__global__ __launch_bounds__(256) void k_cell_from_aos(const double *src, int m, long nstride, long c0, double *dst, long n)
{
    long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    for (int a = 0; a < m; a++) dst[a * nstride + c0 + q] = src[q * m + a];
}
__global__ __launch_bounds__(256) void k_fill(double *p, double v, long n)
{
    long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q < n) p[q] = v;
}

inline unsigned nblk(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

// ============================================================ host context
// the runtime calls of copyout.hpp
struct HipCopy {
    using Error = hipError_t;
    using Event = hipEvent_t;
    using Stream = hipStream_t;
    using Thread = std::thread;
    static constexpr Error OK = hipSuccess;
    static Error alloc(char **p, size_t n) { return hipHostMalloc((void **)p, n, hipHostMallocDefault); }
    static void release(char *p) { (void)hipHostFree(p); }
    static Error event_create(Event *e) { return hipEventCreateWithFlags(e, hipEventDisableTiming); }
    static void event_destroy(Event e) { (void)hipEventDestroy(e); }
    static Error event_record(Event e, Stream st) { return hipEventRecord(e, st); }
    static Error event_wait(Event e) { return hipEventSynchronize(e); }
    static Error to_host(void *dst, const void *src, size_t n, Stream st) { return hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, st); }
    static Error stream_wait(Stream st) { return hipStreamSynchronize(st); }
    // memory the runtime knows nothing of (a failed launch before is left for its own check to report)
    static bool pageable(const void *p)
    {
        if (hipPeekAtLastError() != hipSuccess) return true;
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
        (void)hipGetLastError();
        return true;
    }
    static int device() { int d = 0; (void)hipGetDevice(&d); return d; }
    static void set_device(int d) { (void)hipSetDevice(d); }
    static void clear_error() { (void)hipGetLastError(); }
};

struct cav3d_ctx {
    cav3d_params prm;
    Par P;
    DS S;
    int nb = 0, npv = 0, ntv = 0, ngrd = 0;
    std::vector<BlkD> blk;
    std::vector<std::vector<Seg>> segs = std::vector<std::vector<Seg>>(3);
    std::vector<Con> cons;
    std::vector<std::vector<int>> bcdesc;   // per block: nbc*7 raw
    hipStream_t st = nullptr;
    // the adjoint's cell sources run on another stream, forked from and
    // joined back to st by events (default priority, like st)
    hipStream_t side = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
    int dev = 0;              // device current at creation (the context's device)
    double *stage = nullptr;
    size_t stage_n = 0;
    CopyRing<HipCopy> ring;   // results to the caller (copy_out)
    int nwg_update = 0;
    int sweep_blocks = 0;     // grid of the sweep kernels: as many workgroups as fit the device at once
    int *tiles = nullptr;     // tile table of the sweeps (device): block, j0, k0, diagonal
    int ntiles = 0;
    int *sweep_err = nullptr; // set when a sweep wait gave up
    int *ticket = nullptr;    // next tile of the forward and the backward sweep
    bool profile = false;
    hipEvent_t ev[14] = {};
    double prof_ms[10] = {};  // [8] last cav3d_rhs_vjp, [9] last cav3d_calrhs (device ms)
    std::vector<void *> allocs;
    // grid from vertex coordinates (cav3d_set_grid / cav3d_build_metrics)
    std::vector<std::vector<int>> condesc;   // per block: ncon*22 raw
    double *xv = nullptr;     // vertices, SoA [3][NV], block b from v0[b]
    long NV = 0;
    std::vector<long> v0;
    std::vector<char> has_x;
    double *xc = nullptr;     // cell centroids grd(2:4), SoA [3][NW]
    double *xbuf = nullptr;   // interface-exchange staging
    long xbuf_n = 0;
    // adjoint work arrays (allocated by the first cav3d_rhs_vjp)
    bool adj_ready = false;
    double *a_rb = nullptr, *a_w[3] = {}, *a_snb[3] = {}, *a_fp[3] = {}, *a_vb[3] = {}, *a_vp[3] = {}, *a_ub[3] = {}, *a_mtb[3] = {},
           *a_cb = nullptr, *a_cdb = nullptr, *a_csb = nullptr, *a_pb = nullptr, *a_pbd = nullptr, *a_sum = nullptr, *a_save = nullptr, *a_obj = nullptr;
    int *a_cell[3] = {}, *a_tiles[3] = {}, a_ntiles[3] = {}, a_small = 0;
    long a_obj_n = 0;
};

namespace {

template <class T> int dalloc(cav3d_ctx *c, T **p, size_t n)
{
    *p = nullptr;
    if (n == 0) n = 1;
    HIPCHK(hipMalloc((void **)p, n * sizeof(T)));
    c->allocs.push_back(*p);
    HIPCHK(hipMemsetAsync(*p, 0, n * sizeof(T), c->st));
    return 0;
}

int ensure_stage(cav3d_ctx *c, size_t n)
{
    if (c->stage_n >= n) return 0;
    if (c->stage) { HIPCHK(hipStreamSynchronize(c->st)); HIPCHK(hipFree(c->stage)); c->stage = nullptr; }
    HIPCHK(hipMalloc((void **)&c->stage, n * sizeof(double)));
    c->stage_n = n;
    return 0;
}

int copy_out(cav3d_ctx *c, void *dst, const void *src, size_t bytes, bool wait = true)
{
    const hipError_t e = c->ring.copy(c->st, c->dev, dst, src, bytes, wait);
    return e == hipSuccess ? 0 : fail(std::string("copy to the host: ") + hipGetErrorString(e), -3);
}

int wall_fn(int iturb) { return iturb == 0 ? FN_WALLVISKW : (iturb == -2 ? FN_WALLVIS : FN_WALLINV); }
void set3(int *a, int x, int y, int z) { a[0] = x; a[1] = y; a[2] = z; }

// BC construction (src/bc_module.f90:157-336 faces, :502-866 edges, :870-1185 corners)
int build_bcs(cav3d_ctx *c)
{
    const int iturb = c->prm.iturb;
    for (int w = 0; w < 3; w++) c->segs[w].clear();
    for (int b = 0; b < c->nb; b++) {
        const BlkD &B = c->blk[b];
        const std::vector<int> &dsc = c->bcdesc[b];
        int nbc = (int)dsc.size() / 7;
        std::vector<Seg> faces;
        for (int n = 0; n < nbc; n++) {
            Seg s;
            memset(&s, 0, sizeof(s));
            s.b = b;
            int kind = dsc[7 * n] & CAV3D_BC_KIND_MASK;
            for (int d = 0; d < 3; d++) { s.is[d] = dsc[7 * n + 1 + d]; s.ie[d] = dsc[7 * n + 4 + d]; }
            if (s.is[0] == s.ie[0]) {
                set3(s.dir, -1, 1, 1);
                if (s.is[0] == 1) { s.face = F_IMIN; s.is[0] -= 2; s.org[0] = 2 * s.ie[0] + 1; }
                else { s.face = F_IMAX; s.ie[0] += 2; s.org[0] = 2 * s.is[0] - 1; }
            } else if (s.is[1] == s.ie[1]) {
                set3(s.dir, 1, -1, 1);
                if (s.is[1] == 1) { s.face = F_JMIN; s.is[1] -= 2; s.org[1] = 2 * s.ie[1] + 1; }
                else { s.face = F_JMAX; s.ie[1] += 2; s.org[1] = 2 * s.is[1] - 1; }
            } else if (s.is[2] == s.ie[2]) {
                set3(s.dir, 1, 1, -1);
                if (s.is[2] == 1) { s.face = F_KMIN; s.is[2] -= 2; s.org[2] = 2 * s.ie[2] + 1; }
                else { s.face = F_KMAX; s.ie[2] += 2; s.org[2] = 2 * s.is[2] - 1; }
            } else return fail("boundary range of block " + std::to_string(b) + " is not a face", -2);
            switch (kind) {
            case CAV3D_BC_WALL: s.fn = wall_fn(iturb); break;
            case CAV3D_BC_INFLOW_SUBSONIC: s.fn = FN_INSUB; break;
            case CAV3D_BC_OUTFLOW_SUBSONIC: s.fn = FN_OUTSUB; break;
            case CAV3D_BC_FARFIELD: s.fn = FN_FARFIELD; break;
            case CAV3D_BC_SYMMETRY: s.fn = FN_SYM; break;
            case CAV3D_BC_INFLOW_SUPERSONIC: s.fn = FN_INSUPER; break;
            case CAV3D_BC_OUTFLOW_SUPERSONIC: case CAV3D_BC_DEGENERATE: s.fn = FN_COPY; break;
            case CAV3D_BC_INFLOW: case CAV3D_BC_OUTFLOW: s.fn = FN_EMPTY; break;
            default: return fail("unknown boundary kind " + std::to_string(kind), -2);
            }
            s.pad = kind;
            {
                // the face's own axis spans its three ghost layers; the others stay on interior cells
                const int ext[3] = {B.I, B.J, B.K};
                const int ax = (s.face == F_IMIN || s.face == F_IMAX) ? 0 : ((s.face == F_JMIN || s.face == F_JMAX) ? 1 : 2);
                for (int d = 0; d < 3; d++) {
                    const int lo = (d == ax) ? -1 : 2, hi = (d == ax) ? ext[d] + 3 : ext[d];
                    if (s.is[d] < lo || s.ie[d] > hi || s.is[d] > s.ie[d])
                        return fail("boundary range of block " + std::to_string(b) + " lies outside its face", -2);
                }
            }
            faces.push_back(s);
        }
        auto covers = [&](const int *p, int d0, int d1, int d2) {
            for (const Seg &s : faces) {
                if (s.pad != CAV3D_BC_WALL && s.pad != CAV3D_BC_SYMMETRY) continue;
                bool ok = s.is[d0] <= p[d0] && s.ie[d0] >= p[d0] && s.is[d1] <= p[d1] && s.ie[d1] >= p[d1];
                if (d2 >= 0) ok = ok && s.is[d2] <= p[d2] && s.ie[d2] >= p[d2];
                if (ok) return true;
            }
            return false;
        };
        int I = B.I, J = B.J, K = B.K;
        Seg e[12];
        memset(e, 0, sizeof(e));
        set3(e[0].is, -1, -1, 2); set3(e[0].ie, 1, 1, K); set3(e[0].nb[0], 1, 2, 0); set3(e[0].nb[1], 2, 1, 0); set3(e[0].org, 2, 2, 0);
        set3(e[1].is, I + 1, -1, 2); set3(e[1].ie, I + 3, 1, K); set3(e[1].nb[0], I + 1, 2, 0); set3(e[1].nb[1], I, 1, 0); set3(e[1].org, I, 2, 0);
        set3(e[2].is, -1, J + 1, 2); set3(e[2].ie, 1, J + 3, K); set3(e[2].nb[0], 1, J, 0); set3(e[2].nb[1], 2, J + 1, 0); set3(e[2].org, 2, J, 0);
        set3(e[3].is, I + 1, J + 1, 2); set3(e[3].ie, I + 3, J + 3, K); set3(e[3].nb[0], I + 1, J, 0); set3(e[3].nb[1], I, J + 1, 0); set3(e[3].org, I, J, 0);
        set3(e[4].is, -1, 2, -1); set3(e[4].ie, 1, J, 1); set3(e[4].nb[0], 1, 0, 2); set3(e[4].nb[2], 2, 0, 1); set3(e[4].org, 2, 0, 2);
        set3(e[5].is, I + 1, 2, -1); set3(e[5].ie, I + 3, J, 1); set3(e[5].nb[0], I + 1, 0, 2); set3(e[5].nb[2], I, 0, 1); set3(e[5].org, I, 0, 2);
        set3(e[6].is, -1, 2, K + 1); set3(e[6].ie, 1, J, K + 3); set3(e[6].nb[0], 1, 0, K); set3(e[6].nb[2], 2, 0, K + 1); set3(e[6].org, 2, 0, K);
        set3(e[7].is, I + 1, 2, K + 1); set3(e[7].ie, I + 3, J, K + 3); set3(e[7].nb[0], I + 1, 0, K); set3(e[7].nb[2], I, 0, K + 1); set3(e[7].org, I, 0, K);
        set3(e[8].is, 2, -1, -1); set3(e[8].ie, I, 1, 1); set3(e[8].nb[1], 0, 1, 2); set3(e[8].nb[2], 0, 2, 1); set3(e[8].org, 0, 2, 2);
        set3(e[9].is, 2, J + 1, -1); set3(e[9].ie, I, J + 3, 1); set3(e[9].nb[1], 0, J + 1, 2); set3(e[9].nb[2], 0, J, 1); set3(e[9].org, 0, J, 2);
        set3(e[10].is, 2, -1, K + 1); set3(e[10].ie, I, 1, K + 3); set3(e[10].nb[1], 0, 1, K); set3(e[10].nb[2], 0, 2, K + 1); set3(e[10].org, 0, 2, K);
        set3(e[11].is, 2, J + 1, K + 1); set3(e[11].ie, I, J + 3, K + 3); set3(e[11].nb[1], 0, J + 1, K); set3(e[11].nb[2], 0, J, K + 1); set3(e[11].org, 0, J, K);
        const int ww = iturb == 0 ? FN_EDGEWWKW : FN_EDGEWW;
        for (int m = 0; m < 12; m++) { e[m].b = b; e[m].face = F_NONE; }
        for (int m = 0; m < 4; m++) {
            bool is = covers(e[m].nb[0], 0, 1, -1), js = covers(e[m].nb[1], 0, 1, -1);
            if (is && js) e[m].fn = ww;
            else if (is) { e[m].face = (m == 0 || m == 2) ? F_IMIN : F_IMAX; e[m].org[0] = e[m].nb[1][0]; e[m].org[1] = e[m].nb[1][1]; e[m].fn = wall_fn(iturb); }
            else if (js) { e[m].face = (m == 0 || m == 1) ? F_JMIN : F_JMAX; e[m].org[0] = e[m].nb[0][0]; e[m].org[1] = e[m].nb[0][1]; e[m].fn = wall_fn(iturb); }
            else e[m].fn = FN_EDGENOWALL;
            set3(e[m].dir, 0, 0, 1);
        }
        for (int m = 4; m < 8; m++) {
            bool is = covers(e[m].nb[0], 0, 2, -1), ks = covers(e[m].nb[2], 0, 2, -1);
            if (is && ks) e[m].fn = ww;
            else if (is) { e[m].face = (m == 4 || m == 6) ? F_IMIN : F_IMAX; e[m].org[0] = e[m].nb[2][0]; e[m].org[2] = e[m].nb[2][2]; e[m].fn = wall_fn(iturb); }
            else if (ks) { e[m].face = (m == 4 || m == 5) ? F_KMIN : F_KMAX; e[m].org[0] = e[m].nb[0][0]; e[m].org[2] = e[m].nb[0][2]; e[m].fn = wall_fn(iturb); }
            else e[m].fn = FN_EDGENOWALL;
            set3(e[m].dir, 0, 1, 0);
        }
        for (int m = 8; m < 12; m++) {
            bool js = covers(e[m].nb[1], 1, 2, -1), ks = covers(e[m].nb[2], 1, 2, -1);
            if (js && ks) e[m].fn = ww;
            else if (js) { e[m].face = (m == 8 || m == 10) ? F_JMIN : F_JMAX; e[m].org[1] = e[m].nb[2][1]; e[m].org[2] = e[m].nb[2][2]; e[m].fn = wall_fn(iturb); }
            else if (ks) { e[m].face = (m == 8 || m == 9) ? F_KMIN : F_KMAX; e[m].org[1] = e[m].nb[1][1]; e[m].org[2] = e[m].nb[1][2]; e[m].fn = wall_fn(iturb); }
            else e[m].fn = FN_EDGENOWALL;
            set3(e[m].dir, 1, 0, 0);
        }
        Seg q[8];
        memset(q, 0, sizeof(q));
        for (int m = 0; m < 8; m++) {
            int ib = m & 1, jb = (m >> 1) & 1, kb = (m >> 2) & 1;
            int ig = ib ? I + 1 : 1, jg = jb ? J + 1 : 1, kg = kb ? K + 1 : 1;
            int ic = ib ? I : 2, jc = jb ? J : 2, kc = kb ? K : 2;
            int hi[3] = {I + 1, J + 1, K + 1}, bit[3] = {ib, jb, kb};
            for (int d = 0; d < 3; d++) { q[m].is[d] = bit[d] ? hi[d] : -1; q[m].ie[d] = bit[d] ? hi[d] + 2 : 1; }
            set3(q[m].nb[0], ig, jc, kc); set3(q[m].nb[1], ic, jg, kc); set3(q[m].nb[2], ic, jc, kg);
            set3(q[m].org, ic, jc, kc);
            set3(q[m].nb[3], ic, jg, kg); set3(q[m].nb[4], ig, jc, kg); set3(q[m].nb[5], ig, jg, kc);
            q[m].face = F_NONE;
            q[m].b = b;
        }
        set3(q[5].nb[2], I, 1, K + 1);   // neighbor3 of corner 6 as tabulated at src/bc_module.f90:958-960
        for (int m = 0; m < 8; m++) {
            Seg &cm = q[m];
            bool is = covers(cm.nb[0], 0, 1, 2), js = covers(cm.nb[1], 0, 1, 2), ks = covers(cm.nb[2], 0, 1, 2);
            if (is && js && ks) cm.fn = iturb == 0 ? FN_CORNERWWKW : FN_CORNERWW;
            else if (!is && js && ks) { memcpy(cm.org, cm.nb[0], 12); set3(cm.nb[0], 0, 0, 0); memcpy(cm.nb[1], cm.nb[4], 12); memcpy(cm.nb[2], cm.nb[5], 12); cm.fn = ww; }
            else if (is && !js && ks) { memcpy(cm.org, cm.nb[1], 12); memcpy(cm.nb[0], cm.nb[3], 12); set3(cm.nb[1], 0, 0, 0); memcpy(cm.nb[2], cm.nb[5], 12); cm.fn = ww; }
            else if (is && js && !ks) { memcpy(cm.org, cm.nb[2], 12); memcpy(cm.nb[0], cm.nb[3], 12); memcpy(cm.nb[1], cm.nb[4], 12); set3(cm.nb[2], 0, 0, 0); cm.fn = ww; }
            else if (!is && !js && ks) { cm.face = m < 4 ? F_KMIN : F_KMAX; memcpy(cm.org, cm.nb[5], 12); cm.fn = wall_fn(iturb); }
            else if (is && !js && !ks) { cm.face = (m % 2 == 0) ? F_IMIN : F_IMAX; memcpy(cm.org, cm.nb[3], 12); cm.fn = wall_fn(iturb); }
            else if (!is && js && !ks) { cm.face = (m == 0 || m == 1 || m == 4 || m == 5) ? F_JMIN : F_JMAX; memcpy(cm.org, cm.nb[4], 12); cm.fn = wall_fn(iturb); }
            else cm.fn = FN_CORNERNOWALL;
        }
        for (Seg &s : faces) if (s.fn != FN_EMPTY) c->segs[0].push_back(s);
        for (int m = 0; m < 12; m++) c->segs[1].push_back(e[m]);
        for (int m = 0; m < 8; m++) c->segs[2].push_back(q[m]);
    }
    for (int w = 0; w < 3; w++) {
        long start = 0;
        for (Seg &s : c->segs[w]) {
            s.start = start;
            start += (long)(s.ie[0] - s.is[0] + 1) * (s.ie[1] - s.is[1] + 1) * (s.ie[2] - s.is[2] + 1);
        }
        c->S.NBC[w] = start;
        c->S.nbcseg[w] = (int)c->segs[w].size();
    }
    return 0;
}

// begun: after k_begin, which has done the faces and left the time step's minimum
int launch_setbc(cav3d_ctx *c, bool begun = false)
{
    DS &S = c->S;
    if (S.NBC[0] && !begun) hipLaunchKernelGGL(k_bc, dim3(nblk(S.NBC[0], 128)), dim3(128), 0, c->st, S, 0, 0);
    if (S.NHALO) hipLaunchKernelGGL(k_halo, dim3(nblk(S.NHALO, 128)), dim3(128), 0, c->st, S);
    // (every block has its edges and corners)
    hipLaunchKernelGGL(k_bc, dim3(nblk(S.NBC[1], 128)), dim3(128), 0, c->st, S, 1, begun ? 1 : 0);
    hipLaunchKernelGGL(k_bc, dim3(nblk(S.NBC[2], 128)), dim3(128), 0, c->st, S, 2, 0);
    return 0;
}

int launch_rhs(cav3d_ctx *c)
{
    DS &S = c->S;
    const bool sensor = S.P.nscheme == 2 || S.P.nscheme == 3;
    // AUSMPW+ stays FP64 in the mixed mode: its pressure weight
    // (p + p_ref + rho c^2)/(rho c^2) - 1 is ~1e-5 in water and cancels in FP32
    const bool mixed = c->prm.precision == CAV3D_MIXED && S.P.nscheme != 3;
    FluxWgs g = {};                      // workgroups, each inside one block
    unsigned nc = 0;
    for (const BlkD &B : c->blk) {
        for (int d = 0; d < 3; d++) g.n[d] += nblk(B.nf[d], BLK_WG);
        nc += nblk(B.nc, BLK_WG);
    }
    const bool visc = c->prm.iturb >= -2;
    const dim3 grid((g.n[0] + g.n[1] + g.n[2]) * (visc ? 2 : 1)), block(BLK_WG);
    if (sensor && mixed) hipLaunchKernelGGL((k_face<0, true, float>), grid, block, 0, c->st, S, g);
    else if (sensor && c->prm.precision == CAV3D_MIXED) hipLaunchKernelGGL((k_face<1, true, double>), grid, block, 0, c->st, S, g);
    else if (sensor) hipLaunchKernelGGL((k_face<0, true, double>), grid, block, 0, c->st, S, g);
    else if (mixed) hipLaunchKernelGGL((k_face<0, false, float>), grid, block, 0, c->st, S, g);
    else hipLaunchKernelGGL((k_face<0, false, double>), grid, block, 0, c->st, S, g);
    if (S.P.ncav >= 2 || S.P.ides > 0) hipLaunchKernelGGL(k_combine<true>, dim3(nc), dim3(BLK_WG), 0, c->st, S);
    else hipLaunchKernelGGL(k_combine<false>, dim3(nc), dim3(BLK_WG), 0, c->st, S);
    return 0;
}

int launch_timestep(cav3d_ctx *c)
{
    DS &S = c->S;
    const hipStream_t st = c->st;
    hipLaunchKernelGGL(k_timestep, dim3(nblk(S.NC, 256)), dim3(256), 0, st, S);
    if (c->prm.local == 0) hipLaunchKernelGGL(k_dt_fill, dim3(nblk(S.NC, 256)), dim3(256), 0, st, S);
    hipLaunchKernelGGL(k_time_acc, dim3(1), dim3(64), 0, st, S);
    return 0;
}

// the sweeps' exchange arrays back to "not yet written"
int launch_sweep_fills(cav3d_ctx *c)
{
    DS &S = c->S;
    const long nq = (long)NPV * S.NW;
    hipLaunchKernelGGL(k_sweep_reset, dim3(nblk(nq, 256)), dim3(256), 0, c->st, S, nq, c->ticket);
    return 0;
}

// the face boundaries, the time step and the sweep resets
int launch_begin(cav3d_ctx *c)
{
    DS &S = c->S;
    const long nq = (long)NPV * S.NW;
    const unsigned nbc = nblk(S.NBC[0], 256), nts = nblk(S.NC, 256);
    hipLaunchKernelGGL(k_begin, dim3(nbc + nts + nblk(nq, 256)), dim3(256), 0, c->st, S, nbc, nts, nq, c->ticket);
    return 0;
}

int launch_sweeps(cav3d_ctx *c)
{
    DS &S = c->S;
    const unsigned wz = nblk(S.NC, 128);
    hipLaunchKernelGGL(k_lhs_prep, dim3(wz + nblk(S.NPLANE + 1, ZERO_ROWS)), dim3(128), 0, c->st, S, wz);
    const dim3 grid(c->sweep_blocks), block(SWEEP_THREADS);
    if (c->profile) hipEventRecord(c->ev[6], c->st);
    hipLaunchKernelGGL(k_sweep_tile<true>, grid, block, 0, c->st, S, (const int *)c->tiles, c->ntiles, c->sweep_err, c->ticket);
    if (c->profile) hipEventRecord(c->ev[7], c->st);
    hipLaunchKernelGGL(k_sweep_tile<false>, grid, block, 0, c->st, S, (const int *)c->tiles, c->ntiles, c->sweep_err, c->ticket + 1);
    if (c->profile) hipEventRecord(c->ev[8], c->st);
    return 0;
}

int launch_update(cav3d_ctx *c)
{
    DS &S = c->S;
    hipLaunchKernelGGL(k_update, dim3(c->nwg_update), dim3(256), 0, c->st, S);
    // the final norm reduction beside the eddy viscosity, which reads nothing of it
    hipLaunchKernelGGL(k_finish, dim3(1 + (c->prm.iturb == 0 ? nblk(S.NC, 256) : 0)), dim3(256), 0, c->st, S, c->nwg_update);
    return 0;
}

// a sweep whose bounded wait gave up leaves a flag; report it (stream synchronised by the caller)
int sweep_status(cav3d_ctx *c)
{
    int e = 0;
    HIPCHK(hipMemcpy(&e, c->sweep_err, sizeof(int), hipMemcpyDeviceToHost));
    if (e) return fail("LU-SGS sweep: a dependency wait reached its limit; results of that iteration are invalid", -5);
    return 0;
}

int check_launch(const char *what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(std::string(what) + ": " + hipGetErrorString(e), -3);
    return 0;
}

}  // namespace

// ============================================================ C ABI
extern "C" {

const char *cav3d_last_error(void) { return g_err.c_str(); }

int cav3d_create(const cav3d_params *prm, int nblocks, const cav3d_block *blocks, cav3d_ctx **out)
{
    if (!prm || !blocks || !out) return fail("null argument", -1);
    *out = nullptr;
    if (nblocks < 1 || nblocks > MAXB) return fail("nblocks must be 1.." + std::to_string(MAXB), -1);
    if (prm->iturb != 0 && prm->iturb != -2 && prm->iturb != -3)
        return fail("iturb must be 0 (k-omega SST), -2 (laminar) or -3 (Euler)", -1);
    if (prm->nscheme < 1 || prm->nscheme > 4)
        return fail("nscheme must be 1 (Roe), 2 (Roe-M), 3 (AUSMPW+) or 4 (AUSM+-up)", -1);
    if (prm->nmuscl < 0 || prm->nmuscl > 2 || prm->nlim < 0 || prm->nlim > 10) return fail("bad nmuscl/nlim", -1);
    if (prm->ides < 0 || prm->ides > 4) return fail("ides must be 0 (RANS), 1 (DES), 2 (DDES), 3 (IDDES) or 4 (S-IDDES)", -1);
    if (prm->ncav < 0 || prm->ncav > 5)
        return fail("ncav must be 0 (none), 1 (Merkle), 2 (Kunz), 3 (Singhal), 4 (Schnerr-Sauer) or 5 (Lee)", -1);
    if (prm->cav_clip != 0 && prm->cav_clip != 1) return fail("cav_clip must be 0 (as written) or 1 (species)", -1);
    if (prm->nsteady < 0 || prm->nsteady > 2) return fail("nsteady must be 0, 1 or 2", -1);
    if (!(prm->dt_phy > 0.0)) return fail("dt_phy must be > 0 (it divides the BDF term of getx)", -1);
    if (prm->precision != CAV3D_FP64 && prm->precision != CAV3D_MIXED)
        return fail("precision must be CAV3D_FP64 (0) or CAV3D_MIXED (1)", -1);
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail("no HIP device", -4);
    cav3d_ctx *c = new cav3d_ctx();
    hipGetDevice(&c->dev);
    c->prm = *prm;
    c->nb = nblocks;
    c->npv = prm->iturb == 0 ? 9 : 7;
    c->ntv = prm->iturb == 0 ? 3 : (prm->iturb == -2 ? 2 : 0);
    c->ngrd = prm->iturb == 0 ? 5 : 4;
    Par &P = c->P;
    memset(&P, 0, sizeof(P));
    P.npv = c->npv; P.ntv = c->ntv; P.iturb = prm->iturb; P.nscheme = prm->nscheme; P.nmuscl = prm->nmuscl;
    P.nlim = prm->nlim; P.local = prm->local; P.prec = prm->prec; P.ncav = prm->ncav; P.nsteady = prm->nsteady;
    P.cav_clip = prm->cav_clip;
    P.ides = prm->iturb == 0 ? prm->ides : 0;
    P.cfl = prm->cfl; P.pref = prm->pref; P.uref = prm->uref; P.str = prm->str; P.dt_phy = prm->dt_phy;
    P.c_v = prm->c_v; P.c_c = prm->c_c; P.dp_ref = prm->dp_ref; P.t_ref = prm->t_ref; P.t_crit = prm->t_crit;
    for (int q = 0; q < 9; q++) P.bc_pv[q] = prm->bc_pv[q];
    P.bc_pressure = prm->bc_pressure;
    P.emutref = prm->emutref;
    P.bdf_b = prm->nsteady == 1 ? 1.0 : (prm->nsteady == 2 ? 1.5 * 0.5 : 0.0);
    if (hipStreamCreate(&c->st) != hipSuccess) { delete c; return fail("hipStreamCreate failed", -3); }
    if (hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&c->join, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&c->fork, hipEventDisableTiming) != hipSuccess) {
        cav3d_destroy(c);
        return fail("stream set-up failed", -3);
    }
    DS &S = c->S;
    memset(&S, 0, sizeof(S));
    S.nb = nblocks;
    S.npv = c->npv;
    S.P = P;
    long g0 = 0, c0 = 0, w0 = 0, f0[3] = {0, 0, 0}, x0 = 0, e0 = 0, t0 = 0, p0 = 0;
    c->blk.resize(nblocks);
    c->bcdesc.resize(nblocks);
    for (int b = 0; b < nblocks; b++) {
        const cav3d_block &cb = blocks[b];
        if (cb.imax < 4 || cb.jmax < 4 || cb.kmax < 4) { delete c; return fail("each block needs at least 3 cells per direction", -1); }
        BlkD &B = c->blk[b];
        B.I = cb.imax; B.J = cb.jmax; B.K = cb.kmax;
        B.nx = B.I + 5; B.ny = B.J + 5;
        B.ng = (long)B.nx * B.ny * (B.K + 5);
        B.nc = (long)(B.I - 1) * (B.J - 1) * (B.K - 1);
        B.nw = (long)(B.I + 1) * (B.J + 1) * (B.K + 1);
        B.nf[0] = (long)B.I * (B.J - 1) * (B.K - 1);
        B.nf[1] = (long)(B.I - 1) * B.J * (B.K - 1);
        B.nf[2] = (long)(B.I - 1) * (B.J - 1) * B.K;
        B.ncx = (long)B.I * (B.J + 1) * (B.K + 1);
        B.nex = (long)(B.I + 1) * B.J * (B.K + 1);
        B.ntx = (long)(B.I + 1) * (B.J + 1) * B.K;
        B.g0 = g0; B.c0 = c0; B.w0 = w0; B.cx0 = x0; B.ex0 = e0; B.tx0 = t0;
        for (int d = 0; d < 3; d++) { B.f0[d] = f0[d]; f0[d] += B.nf[d]; }
        B.p0 = p0;
        p0 += (long)(B.J - 1) * (B.K - 1);
        g0 += B.ng; c0 += B.nc; w0 += B.nw; x0 += B.ncx; e0 += B.nex; t0 += B.ntx;
        S.b[b] = B;
        if (cb.nbc < 0 || (cb.nbc > 0 && !cb.bc)) { delete c; return fail("bad bc list", -1); }
        c->bcdesc[b].assign(cb.bc, cb.bc + 7 * cb.nbc);
    }
    S.NG = g0; S.NC = c0; S.NW = w0; S.NCX = x0; S.NEX = e0; S.NTX = t0; S.NPLANE = p0;
    for (int d = 0; d < 3; d++) S.NF[d] = f0[d];
    // interfaces
    long hs = 0;
    c->condesc.resize(nblocks);
    for (int b = 0; b < nblocks; b++) {
        const cav3d_block &cb = blocks[b];
        if (cb.ncon < 0 || (cb.ncon > 0 && !cb.con)) { delete c; return fail("bad interface list", -1); }
        c->condesc[b].assign(cb.con, cb.con + 22 * cb.ncon);
        for (int n = 0; n < cb.ncon; n++) {
            const int *d = cb.con + 22 * n;
            Con cn;
            memset(&cn, 0, sizeof(cn));
            cn.src = b; cn.dst = d[0];
            if (cn.dst < 0 || cn.dst >= nblocks) { delete c; return fail("interface donor out of range", -1); }
            for (int q = 0; q < 3; q++) { cn.is[q] = d[1 + q]; cn.ie[q] = d[4 + q]; cn.isd[q] = d[7 + q]; }
            for (int q = 0; q < 9; q++) cn.tm[q] = d[13 + q];
            long cnt = 1;
            for (int q = 0; q < 3; q++) cnt *= (cn.ie[q] >= cn.is[q]) ? (cn.ie[q] - cn.is[q] + 1) : 0;
            if (cnt == 0) continue;
            // both the source box and its image must lie inside the ghosted arrays
            const int ext[2][3] = {{blocks[b].imax, blocks[b].jmax, blocks[b].kmax},
                                   {blocks[cn.dst].imax, blocks[cn.dst].jmax, blocks[cn.dst].kmax}};
            bool ok = true;
            for (int q = 0; q < 3; q++) {
                if (cn.is[q] < -1 || cn.ie[q] > ext[0][q] + 3) ok = false;
                for (int r = 0; r < 3; r++)
                    if (cn.tm[3 * q + r] < -1 || cn.tm[3 * q + r] > 1) ok = false;
            }
            for (int corner = 0; ok && corner < 8; corner++) {
                int del[3];
                for (int q = 0; q < 3; q++) del[q] = ((corner >> q) & 1) ? cn.ie[q] - cn.is[q] : 0;
                for (int q = 0; q < 3; q++) {
                    int v = cn.tm[3 * q] * del[0] + cn.tm[3 * q + 1] * del[1] + cn.tm[3 * q + 2] * del[2] + cn.isd[q];
                    if (v < -1 || v > ext[1][q] + 3) ok = false;
                }
            }
            if (!ok) { delete c; return fail("interface " + std::to_string(n) + " of block " + std::to_string(b) +
                                             " maps outside the ghosted arrays", -1); }
            cn.start = hs;
            hs += cnt;
            c->cons.push_back(cn);
        }
    }
    S.NHALO = hs;
    S.ncon = (int)c->cons.size();
    int rc = build_bcs(c);
    if (rc) { cav3d_destroy(c); return rc; }
    const int npv = c->npv;
    if ((rc = dalloc(c, &S.pv, npv * S.NG)) || (rc = dalloc(c, &S.dc, (long)ND * S.NG)) ||
        (rc = dalloc(c, &S.vol, S.NW)) || (rc = dalloc(c, &c->xc, 3 * S.NW)) || (rc = dalloc(c, &S.cx, 3 * S.NCX)) || (rc = dalloc(c, &S.ex, 3 * S.NEX)) ||
        (rc = dalloc(c, &S.tx, 3 * S.NTX)) || (rc = dalloc(c, &S.res, npv * S.NC)) || (rc = dalloc(c, &S.dt, S.NC)) ||
        (rc = dalloc(c, &S.img, RC_N * (S.NF[0] + 1))) ||
        (rc = dalloc(c, &S.xqf, (long)NPV * S.NW)) || (rc = dalloc(c, &S.xqb, (long)NPV * S.NW)) ||
        (rc = dalloc(c, &S.scal, 32))) { cav3d_destroy(c); return rc; }
    if (hipMemcpyAsync(S.scal, &DT_NONE, sizeof(DT_NONE), hipMemcpyHostToDevice, c->st) != hipSuccess) {
        cav3d_destroy(c); return fail("device set-up failed", -3);
    }
    // the face fluxes live from the faces to the combine, the records from
    // k_lhs_prep behind it to the backward sweep: they share their memory (18
    // numbers a face, of which there are at most 4 to a cell where a block
    // has 3 cells a direction, against RC_N a cell)
    static_assert(2 * NPV * 4 <= RC_N, "the fluxes fit the records' memory");
    S.ff[0] = S.img;
    for (int d = 1; d < 3; d++) S.ff[d] = S.ff[d - 1] + 2 * npv * S.NF[d - 1];
    if (prm->iturb == 0) {
        if ((rc = dalloc(c, &S.mut, S.NG)) || (rc = dalloc(c, &S.ydn, S.NW)) || (rc = dalloc(c, &S.itt, 4 * S.NC)) ||
            (rc = dalloc(c, &S.ocut, S.NC))) { cav3d_destroy(c); return rc; }
    }
    if (prm->ncav) {
        if ((rc = dalloc(c, &S.icav, 4 * S.NC)) || (rc = dalloc(c, &S.rcav, 2 * S.NC))) { cav3d_destroy(c); return rc; }
    }
    if (prm->nsteady > 0) {
        if ((rc = dalloc(c, &S.qq, 2 * npv * S.NC))) { cav3d_destroy(c); return rc; }
    }
    {
        // tile table: TJ x TK pencil tiles of every block, ordered by the tile
        // diagonal tj + tk (the forward sweep takes them in this order, the
        // backward sweep in reverse)
        std::vector<std::array<int, 4>> tl;
        for (int b = 0; b < nblocks; b++) {
            const int ntj = (c->blk[b].J - 1 + TJ - 1) / TJ, ntk = (c->blk[b].K - 1 + TK - 1) / TK;
            for (int tk = 0; tk < ntk; tk++)
                for (int tj = 0; tj < ntj; tj++) tl.push_back({b, 2 + TJ * tj, 2 + TK * tk, tj + tk});
        }
        std::stable_sort(tl.begin(), tl.end(), [](const std::array<int, 4> &x, const std::array<int, 4> &y) {
            return x[3] < y[3];
        });
        std::vector<int> tab;
        for (auto &t : tl) tab.insert(tab.end(), t.begin(), t.end());
        c->ntiles = (int)tl.size();
        if ((rc = dalloc(c, &c->tiles, tab.size())) || (rc = dalloc(c, &c->sweep_err, 3))) {
            cav3d_destroy(c); return rc;
        }
        c->ticket = c->sweep_err + 1;
        if (hipMemcpyAsync(c->tiles, tab.data(), tab.size() * sizeof(int), hipMemcpyHostToDevice, c->st) != hipSuccess) {
            cav3d_destroy(c); return fail("tile table upload failed", -3);
        }
        int dev = 0, ncu = 0, per = 0, per2 = 0;
        hipGetDevice(&dev);
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void *)k_sweep_tile<true>, SWEEP_THREADS, 0);
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per2, (const void *)k_sweep_tile<false>, SWEEP_THREADS, 0);
        per = std::min(per, per2);
        long cap = (long)ncu * per;
        if (cap < 1) { cav3d_destroy(c); return fail("sweep kernel cannot be made resident", -3); }
        c->sweep_blocks = (int)std::max(1L, std::min((long)c->ntiles, cap));
    }
    c->nwg_update = (int)nblk(S.NC, 256);
    if ((rc = dalloc(c, &S.red, (long)c->nwg_update * (NPV + 2)))) { cav3d_destroy(c); return rc; }
    for (int w = 0; w < 3; w++) {
        if ((rc = dalloc(c, &S.seg[w], c->segs[w].size()))) { cav3d_destroy(c); return rc; }
        if (!c->segs[w].empty() &&
            hipMemcpyAsync(S.seg[w], c->segs[w].data(), c->segs[w].size() * sizeof(Seg), hipMemcpyHostToDevice, c->st) != hipSuccess) {
            cav3d_destroy(c); return fail("segment upload failed", -3);
        }
    }
    if ((rc = dalloc(c, &S.con, c->cons.size()))) { cav3d_destroy(c); return rc; }
    if (!c->cons.empty() &&
        hipMemcpyAsync(S.con, c->cons.data(), c->cons.size() * sizeof(Con), hipMemcpyHostToDevice, c->st) != hipSuccess) {
        cav3d_destroy(c); return fail("interface upload failed", -3);
    }
    for (int q = 0; q < 14; q++) hipEventCreate(&c->ev[q]);
    if (hipStreamSynchronize(c->st) != hipSuccess) { cav3d_destroy(c); return fail("device set-up failed", -3); }
    *out = c;
    return 0;
}

void cav3d_destroy(cav3d_ctx *c)
{
    if (!c) return;
    if (c->st) hipStreamSynchronize(c->st);
    for (void *p : c->allocs) hipFree(p);
    if (c->stage) hipFree(c->stage);
    c->ring.close();
    if (c->xbuf) hipFree(c->xbuf);
    if (c->a_obj) hipFree(c->a_obj);
    for (int q = 0; q < 14; q++) if (c->ev[q]) hipEventDestroy(c->ev[q]);
    if (c->side) { hipStreamSynchronize(c->side); hipStreamDestroy(c->side); }
    if (c->join) hipEventDestroy(c->join);
    if (c->fork) hipEventDestroy(c->fork);
    if (c->st) hipStreamDestroy(c->st);
    delete c;
}

int cav3d_set_metrics(cav3d_ctx *c, int b, const double *cx, const double *ex, const double *tx, const double *grd)
{
    if (!c || b < 0 || b >= c->nb || !cx || !ex || !tx || !grd) return fail("bad argument to cav3d_set_metrics", -1);
    const BlkD &B = c->blk[b];
    DS &S = c->S;
    int rc;
    long nmax = std::max(std::max(3 * B.ncx, 3 * B.nex), std::max(3 * B.ntx, (long)c->ngrd * B.nw));
    if ((rc = ensure_stage(c, nmax))) return rc;
    struct { const double *h; long n; double *d; long nst; long o; } parts[3] = {
        {cx, B.ncx, S.cx, S.NCX, B.cx0}, {ex, B.nex, S.ex, S.NEX, B.ex0}, {tx, B.ntx, S.tx, S.NTX, B.tx0}};
    for (auto &p : parts) {
        HIPCHK(hipMemcpyAsync(c->stage, p.h, 3 * p.n * sizeof(double), hipMemcpyHostToDevice, c->st));
        hipLaunchKernelGGL(k_aos_to_soa, dim3(nblk(p.n, 256)), dim3(256), 0, c->st, (const double *)c->stage, 3, 3, 0, p.d, p.nst, p.o, p.n);
        HIPCHK(hipStreamSynchronize(c->st));
    }
    HIPCHK(hipMemcpyAsync(c->stage, grd, (long)c->ngrd * B.nw * sizeof(double), hipMemcpyHostToDevice, c->st));
    hipLaunchKernelGGL(k_aos_to_soa, dim3(nblk(B.nw, 256)), dim3(256), 0, c->st, (const double *)c->stage, 1, c->ngrd, 0, S.vol, S.NW, B.w0, B.nw);
    hipLaunchKernelGGL(k_aos_to_soa, dim3(nblk(B.nw, 256)), dim3(256), 0, c->st, (const double *)c->stage, 3, c->ngrd, 1, c->xc, S.NW, B.w0, B.nw);
    if (S.ydn)
        hipLaunchKernelGGL(k_aos_to_soa, dim3(nblk(B.nw, 256)), dim3(256), 0, c->st, (const double *)c->stage, 1, c->ngrd, 4, S.ydn, S.NW, B.w0, B.nw);
    HIPCHK(hipStreamSynchronize(c->st));
    return check_launch("cav3d_set_metrics");
}

int cav3d_put_state(cav3d_ctx *c, int b, const double *pv, const double *dv, const double *tv, const double *qq)
{
    if (!c || b < 0 || b >= c->nb || !pv) return fail("bad argument to cav3d_put_state", -1);
    const BlkD &B = c->blk[b];
    DS &S = c->S;
    int rc;
    if ((rc = ensure_stage(c, (long)(18 + 3) * B.ng + 2L * c->npv * B.nc))) return rc;
    HIPCHK(hipMemcpyAsync(c->stage, pv, (long)c->npv * B.ng * sizeof(double), hipMemcpyHostToDevice, c->st));
    hipLaunchKernelGGL(k_aos_to_soa, dim3(nblk(B.ng, 256)), dim3(256), 0, c->st, (const double *)c->stage, c->npv, c->npv, 0, S.pv, S.NG, B.g0, B.ng);
    HIPCHK(hipStreamSynchronize(c->st));
    if (dv) {
        HIPCHK(hipMemcpyAsync(c->stage, dv, 18L * B.ng * sizeof(double), hipMemcpyHostToDevice, c->st));
        double *tvd = c->stage + 18L * B.ng;
        if (tv && c->ntv) HIPCHK(hipMemcpyAsync(tvd, tv, (long)c->ntv * B.ng * sizeof(double), hipMemcpyHostToDevice, c->st));
        hipLaunchKernelGGL(k_dv_to_dc, dim3(nblk(B.ng, 256)), dim3(256), 0, c->st, (const double *)c->stage,
                           (const double *)tvd, (tv ? c->ntv : 0), S.dc, S.mut, S.NG, B.g0, B.ng);
        HIPCHK(hipStreamSynchronize(c->st));
    } else {
        DS S1 = S;   // evaluate this block's interior only
        S1.nb = 1; S1.b[0] = B; S1.b[0].c0 = 0; S1.NC = B.nc;
        S1.b[0].g0 = B.g0;
        hipLaunchKernelGGL(k_eos_cells, dim3(nblk(B.nc, 128)), dim3(128), 0, c->st, S1, 1, 1);
        HIPCHK(hipStreamSynchronize(c->st));
    }
    if (c->prm.nsteady > 0) {
        if (qq) {
            HIPCHK(hipMemcpyAsync(c->stage, qq, 2L * c->npv * B.nc * sizeof(double), hipMemcpyHostToDevice, c->st));
            hipLaunchKernelGGL(k_cell_from_aos, dim3(nblk(B.nc, 256)), dim3(256), 0, c->st, (const double *)c->stage,
                               2 * c->npv, S.NC, B.c0, S.qq, B.nc);
        } else {
            DS S1 = S;
            S1.nb = 1; S1.b[0] = B; S1.NC = S.NC;
            // both levels from the current state (initial_module set_others)
            hipLaunchKernelGGL(k_unsteady_shift, dim3(nblk(S.NC, 256)), dim3(256), 0, c->st, S);
            hipLaunchKernelGGL(k_unsteady_shift, dim3(nblk(S.NC, 256)), dim3(256), 0, c->st, S);
        }
        HIPCHK(hipStreamSynchronize(c->st));
    }
    return check_launch("cav3d_put_state");
}

int cav3d_get_state(cav3d_ctx *c, int b, double *pv, double *dv, double *tv, double *qq)
{
    if (!c || b < 0 || b >= c->nb) return fail("bad argument to cav3d_get_state", -1);
    const BlkD &B = c->blk[b];
    DS &S = c->S;
    int rc;
    HIPCHK(hipStreamSynchronize(c->st));
    if ((rc = ensure_stage(c, (long)(18 + 3) * B.ng + 2L * c->npv * B.nc))) return rc;
    if (pv) {
        hipLaunchKernelGGL(k_soa_to_aos, dim3(nblk(B.ng, 256)), dim3(256), 0, c->st, (const double *)S.pv, c->npv, S.NG, B.g0, c->stage, B.ng);
        if ((rc = copy_out(c, pv, c->stage, (long)c->npv * B.ng * sizeof(double)))) return rc;
    }
    if (dv || tv) {
        // evaluate the EOS over this block's ghosted cells into AoS staging
        double *dvd = c->stage, *tvd = c->stage + 18L * B.ng;
        hipLaunchKernelGGL(k_eos_full, dim3(nblk(B.ng, 128)), dim3(128), 0, c->st, S, B.g0, B.ng, dvd, tvd);
        HIPCHK(hipStreamSynchronize(c->st));
        if (dv && (rc = copy_out(c, dv, dvd, 18L * B.ng * sizeof(double)))) return rc;
        if (tv && c->ntv) {
            std::vector<double> t2(2 * B.ng), mt;
            HIPCHK(hipMemcpy(t2.data(), tvd, 2L * B.ng * sizeof(double), hipMemcpyDeviceToHost));
            if (c->ntv == 3) {
                mt.resize(B.ng);
                HIPCHK(hipMemcpy(mt.data(), S.mut + B.g0, B.ng * sizeof(double), hipMemcpyDeviceToHost));
            }
            for (long g = 0; g < B.ng; g++) {
                tv[c->ntv * g] = t2[2 * g];
                tv[c->ntv * g + 1] = t2[2 * g + 1];
                if (c->ntv == 3) tv[3 * g + 2] = mt[g];
            }
        }
    }
    if (qq && c->prm.nsteady > 0) {
        hipLaunchKernelGGL(k_cell_to_aos, dim3(nblk(B.nc, 256)), dim3(256), 0, c->st, (const double *)S.qq, 2 * c->npv, S.NC, B.c0, c->stage, B.nc);
        if ((rc = copy_out(c, qq, c->stage, 2L * c->npv * B.nc * sizeof(double)))) return rc;
    }
    return check_launch("cav3d_get_state");
}

int cav3d_setbc(cav3d_ctx *c)
{
    if (!c) return fail("null context", -1);
    launch_setbc(c);
    HIPCHK(hipStreamSynchronize(c->st));
    return check_launch("cav3d_setbc");
}

int cav3d_timestep(cav3d_ctx *c, int b, double *dt)
{
    if (!c || b < 0 || b >= c->nb) return fail("bad argument to cav3d_timestep", -1);
    launch_timestep(c);
    const BlkD &B = c->blk[b];
    if (dt) HIPCHK(hipMemcpyAsync(dt, c->S.dt + B.c0, B.nc * sizeof(double), hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    return check_launch("cav3d_timestep");
}

int cav3d_calrhs(cav3d_ctx *c, double time, int b, double *res, double *icav, double *itt, double *omega_cut)
{
    (void)time;
    if (!c || b < 0 || b >= c->nb) return fail("bad argument to cav3d_calrhs", -1);
    DS &S = c->S;
    const BlkD &B = c->blk[b];
    int rc;
    if ((rc = ensure_stage(c, (long)c->npv * B.nc))) return rc;
    if (c->profile) hipEventRecord(c->ev[12], c->st);
    launch_rhs(c);
    if (c->profile) {
        hipEventRecord(c->ev[13], c->st);
        hipEventSynchronize(c->ev[13]);
        float ms;
        hipEventElapsedTime(&ms, c->ev[12], c->ev[13]);
        c->prof_ms[9] = ms;
    }
    struct { double *h; const double *d; int m; } outs[4] = {{res, S.res, c->npv}, {icav, S.icav, 4}, {itt, S.itt, 4}, {omega_cut, S.ocut, 1}};
    for (auto &o : outs) {
        if (!o.h) continue;
        if (!o.d) { memset(o.h, 0, sizeof(double) * o.m * B.nc); continue; }
        hipLaunchKernelGGL(k_cell_to_aos, dim3(nblk(B.nc, 256)), dim3(256), 0, c->st, o.d, o.m, S.NC, B.c0, c->stage, B.nc);
        if ((rc = copy_out(c, o.h, c->stage, (long)o.m * B.nc * sizeof(double)))) return rc;
    }
    HIPCHK(hipStreamSynchronize(c->st));
    return check_launch("cav3d_calrhs");
}

int cav3d_timeinteg(cav3d_ctx *c, int nt_phy, int nt, double timeprev, double *time)
{
    (void)nt;
    if (!c) return fail("null context", -1);
    if (c->profile) hipEventRecord(c->ev[0], c->st);
    // (a time step that all cells share takes another pass over dt)
    const bool begun = c->prm.local != 0;
    if (begun) {
        launch_begin(c);
    } else {
        launch_sweep_fills(c);
        launch_timestep(c);
    }
    if (c->profile) hipEventRecord(c->ev[1], c->st);
    launch_setbc(c, begun);
    if (c->profile) hipEventRecord(c->ev[2], c->st);
    launch_rhs(c);
    if (c->profile) hipEventRecord(c->ev[3], c->st);
    int lrc = launch_sweeps(c);
    if (lrc) return lrc;
    if (c->profile) hipEventRecord(c->ev[4], c->st);
    launch_update(c);
    if (c->profile) {
        hipEventRecord(c->ev[5], c->st);
        hipEventSynchronize(c->ev[5]);
        float ms;
        for (int q = 0; q < 5; q++) { hipEventElapsedTime(&ms, c->ev[q], c->ev[q + 1]); c->prof_ms[q] = ms; }
        hipEventElapsedTime(&ms, c->ev[0], c->ev[5]);
        c->prof_ms[5] = ms;
        hipEventElapsedTime(&ms, c->ev[6], c->ev[7]);
        c->prof_ms[6] = ms;
        hipEventElapsedTime(&ms, c->ev[7], c->ev[8]);
        c->prof_ms[7] = ms;
    }
    int rc = check_launch("cav3d_timeinteg");
    if (rc) return rc;
    if (time) {
        double tacc;
        HIPCHK(hipMemcpyAsync(&tacc, c->S.scal + 1, sizeof(double), hipMemcpyDeviceToHost, c->st));
        HIPCHK(hipStreamSynchronize(c->st));
        if ((rc = sweep_status(c))) return rc;
        *time = (c->prm.nsteady == 0) ? tacc + timeprev : c->prm.dt_phy * (double)nt_phy;
    }
    return 0;
}

int cav3d_residual(cav3d_ctx *c, double *l2, int *ijk, double *resmax)
{
    if (!c) return fail("null context", -1);
    double h[32];
    HIPCHK(hipMemcpyAsync(h, c->S.scal, sizeof(h), hipMemcpyDeviceToHost, c->st));
    HIPCHK(hipStreamSynchronize(c->st));
    int rc = sweep_status(c);
    if (rc) return rc;
    if (l2) for (int n = 0; n < c->npv; n++) l2[n] = h[4 + n];
    long bi;
    memcpy(&bi, &h[5 + NPV], sizeof(long));
    double bm = h[4 + NPV];
    if (ijk) {
        if (bm > 1.0e-12) {
            ijk[0] = (int)(bi >> 48); ijk[1] = (int)(bi & 0xffff); ijk[2] = (int)((bi >> 16) & 0xffff); ijk[3] = (int)((bi >> 32) & 0xffff);
        } else { ijk[0] = -1; ijk[1] = ijk[2] = ijk[3] = 0; }
    }
    if (resmax) *resmax = bm > 1.0e-12 ? bm : 1.0e-12;
    return 0;
}

int cav3d_unsteady_shift(cav3d_ctx *c)
{
    if (!c) return fail("null context", -1);
    if (c->prm.nsteady == 0) return 0;
    hipLaunchKernelGGL(k_unsteady_shift, dim3(nblk(c->S.NC, 256)), dim3(256), 0, c->st, c->S);
    HIPCHK(hipStreamSynchronize(c->st));
    return check_launch("cav3d_unsteady_shift");
}

int cav3d_eos(cav3d_ctx *c, int n, const double *p, const double *t, const double *y1, const double *y2, double *dv, double *tv)
{
    if (!c || n < 0 || !p || !t || !y1 || !y2 || !dv || !tv) return fail("bad argument to cav3d_eos", -1);
    if (n == 0) return 0;
    int rc;
    if ((rc = ensure_stage(c, 24L * n))) return rc;
    double *d = c->stage;
    HIPCHK(hipMemcpyAsync(d, p, n * 8, hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(d + n, t, n * 8, hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(d + 2L * n, y1, n * 8, hipMemcpyHostToDevice, c->st));
    HIPCHK(hipMemcpyAsync(d + 3L * n, y2, n * 8, hipMemcpyHostToDevice, c->st));
    hipLaunchKernelGGL(k_eos_points, dim3(nblk(n, 128)), dim3(128), 0, c->st, c->P, n, (const double *)d, (const double *)(d + n),
                       (const double *)(d + 2L * n), (const double *)(d + 3L * n), d + 4L * n, d + 22L * n);
    if ((rc = copy_out(c, dv, d + 4L * n, 18L * n * 8, false)) || (rc = copy_out(c, tv, d + 22L * n, 2L * n * 8))) return rc;
    return check_launch("cav3d_eos");
}

int cav3d_eos_host(int n, const double *p, const double *t, const double *y1, const double *y2, double *dv, double *tv)
{
    if (n < 0 || !p || !t || !y1 || !y2 || !dv || !tv) return fail("bad argument to cav3d_eos_host", -1);
    auto work = [&](int lo, int hi) {
        for (int q = lo; q < hi; q++) {
            double d[ND];
            mixture_eos<double>(p[q], t[q], y1[q], y2[q], d, true, dv + 18L * q);
            tv[2L * q] = d[D_MU];
            tv[2L * q + 1] = d[D_KAP];
        }
    };
    int nt = (int)std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
    if (n < 4096) nt = 1;
    std::vector<std::thread> th;
    for (int w = 0; w < nt; w++) th.emplace_back(work, (int)((long)n * w / nt), (int)((long)n * (w + 1) / nt));
    for (auto &x : th) x.join();
    return 0;
}

int cav3d_profile(cav3d_ctx *c, int enable, double *out)
{
    if (!c) return fail("null context", -1);
    c->profile = enable != 0;
    if (out) for (int q = 0; q < 10; q++) out[q] = c->prof_ms[q];
    return 0;
}

int cav3d_synchronize(cav3d_ctx *c)
{
    if (!c) return fail("null context", -1);
    HIPCHK(hipStreamSynchronize(c->st));
    return check_launch("cav3d_synchronize");
}

}  // extern "C"

#include "metrics.hpp"
#include "post.hpp"
#include "adjoint.hpp"

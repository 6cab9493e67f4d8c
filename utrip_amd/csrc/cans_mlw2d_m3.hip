// cans_mlw2d_m3.hip -- the 2D step of mlw_m3, the modified Lax-Wendroff
// engine for MHD with all three vector components (cans2d/hdmlw/mlw_m3.f:2-377),
// on gfx950, FP64 bit-identical to the reference compiled without FMA
// contraction.  One launch takes the step, and in a run whose ghost cells are
// copies of interior cells (per_margin > 0) also writes those copies, takes
// the next step's cfl_m3 (cans2d/common/cfl_m3.f:44-62) and advances the clock.
//
// The kernel marches as cans_mlw2d.hip does (strips of 62 columns, a wave
// each, neighbours in x from the adjacent lanes, each row's state handed to
// the next), and is bound by the same thing, FP64 issue with two waves on a
// SIMD.  Its row state is larger: 61 doubles a lane carried and as many more
// within a row do not fit the 256 registers of two waves per SIMD.  So what a
// row leaves for the next only to be subtracted there (cell and corner
// fluxes of the south row, south differences; 31 doubles a lane) waits in LDS
// slots of the lane's own, 15.5 KB a wave and 124 KB a CU, without barriers;
// and each equation is taken in two goes, one that uses up its cell values
// (half step, centred term, viscosity) and one its corner fluxes.
//
// A step with its ghost copies, cfl and clock, periodic boxes, against tiles
// of 31 x 7 cells through LDS (1.4 cells formed per cell stepped, three
// barriers) and a fill pass: 64^2 17.9 -> 11.2 us, 256^2 22.9 -> 17.1, 512^2
// 39.5 -> 26.9, 1024^2 99 -> 54, 2048^2 378 -> 185; no size was better tiled.
#include "cans_clock.hpp"
#include "cans_common.hpp"
#include "cans_kernels.hpp"
#include "cans_march2d.hpp"
#include "cans_wave.hpp"

namespace cans {
using namespace march2d;
namespace {

// u: ro ee rx ry rz bx by bz (mlw_m3.f:107-120)
enum { U_RO, U_EE, U_RX, U_RY, U_RZ, U_BX, U_BY, U_BZ, NU };
// fluxes (mlw_m3.f:121-202), of cells and corners:
//   x: ro*vx eex rxx ryx rzx 0 -ez ey;  y: ro*vy eey rxy ryy rzy ez 0 -ex
struct Cell {
    double u[NU];
    double eex, eey, rxx, rxy, ryx, ryy, rzx, rzy, nex, ey, ez;
    double vx, vy;
};
struct Prim {
    double ro, pr, vx, vy, vz, bx, by, bz;
};

// LDS slots of a lane: from the row below (j-1), the y fluxes of its cell and
// of its corner, the corner x-flux differences, u(i,j)-u(i,j-1), the Az sum
// of the corner row and the viscosity coefficient of face j-1/2
enum { K_SY = 0, K_KY = 7, K_DX = 14, K_DS = 21, K_PS = 29, K_QY = 30, NK = 31 };
enum { W_RO, W_EE, W_RX, W_RY, W_RZ, W_BX, W_BZ, W_BY = W_BX };   // slot order of SY/KY (bx) and DX (by)

CANS_DEV Prim load_prim(const Mlw3Args &a, const ColCtx &x, int j) {
    const int jc = j < 1 ? 1 : (j > a.jx ? a.jx : j);
    const size_t r = (size_t)(jc - 1) * (size_t)a.ix;
    unsigned bo = x.boff;                  // opaque: scalar row base + 32-bit lane offset
    asm volatile("" : "+v"(bo));
    Prim p;
    p.ro = ld(a.in[0] + r, bo); p.pr = ld(a.in[1] + r, bo); p.vx = ld(a.in[2] + r, bo); p.vy = ld(a.in[3] + r, bo);
    p.vz = ld(a.in[4] + r, bo); p.bx = ld(a.in[5] + r, bo); p.by = ld(a.in[6] + r, bo); p.bz = ld(a.in[7] + r, bo);
    return p;
}

CANS_DEV Cell make_cell(const Prim &p, double gm) {
    Cell c;
    const double ro = p.ro, pr = p.pr, vx = p.vx, vy = p.vy, vz = p.vz, bx = p.bx, by = p.by, bz = p.bz;
    const double vv = vx * vx + vy * vy + vz * vz;
    const double bb = bx * bx + by * by + bz * bz;
    c.u[U_RO] = ro;
    c.u[U_EE] = pr / (gm - 1.0) + 0.5 * ro * vv + pi8i * bb;
    c.u[U_RX] = ro * vx;
    c.u[U_RY] = ro * vy;
    c.u[U_RZ] = ro * vz;
    c.u[U_BX] = bx;
    c.u[U_BY] = by;
    c.u[U_BZ] = bz;
    const double ex = -vy * bz + vz * by;
    const double ey = -vz * bx + vx * bz;
    const double ez = -vx * by + vy * bx;
    const double ep = pr * gm / (gm - 1.0) + 0.5 * ro * vv;
    c.eex = ep * vx + (bz * ey - by * ez) * pi4i;
    c.eey = ep * vy + (bx * ez - bz * ex) * pi4i;
    c.rxx = ro * (vx * vx) + pr + pi8i * (by * by + bz * bz - bx * bx);
    c.rxy = ro * vx * vy - pi4i * bx * by;
    c.ryx = ro * vy * vx - pi4i * by * bx;
    c.ryy = ro * (vy * vy) + pr + pi8i * (bx * bx + bz * bz - by * by);
    c.rzx = ro * vz * vx - pi4i * bz * bx;
    c.rzy = ro * vz * vy - pi4i * bz * by;
    c.nex = -ex;
    c.ey = ey;
    c.ez = ez;
    c.vx = vx;
    c.vy = vy;
    return c;
}

// The half step at a corner (mlwhalf.f:45-52): A = (i,j), B = (i+1,j),
// C = (i,j+1), D = (i+1,j+1).  z is the term of a flux that is zero
// everywhere, dt*(+0).
struct Quad {
    double A, B, C, D;
};
CANS_DEV Quad quad(double a, double n) { return Quad{a, shl1(a), n, shl1(n)}; }
CANS_DEV double hx(const Quad &f, double dxim, double dt) { return dt * (dxim * (f.B - f.A + f.D - f.C) / 2.0); }
CANS_DEV double hy(const Quad &g, double dyim, double dt) { return dt * (dyim * (g.C - g.A + g.D - g.B) / 2.0); }
CANS_DEV double hu(const Quad &u) { return 0.25 * (u.B + u.A + u.D + u.C); }

struct Corner {
    double u[NU];      // half-step values
    double rox, roy, eex, eey, rxx, rxy, ryx, ryy, rzx, rzy, nex, ey, ez;
};
// half-step primitives, E and the corner fluxes (mlw_m3.f:214-310)
CANS_DEV void corner_fluxes(Corner &k, double gm) {
    const double roh = k.u[U_RO], eeh = k.u[U_EE], bxh = k.u[U_BX], byh = k.u[U_BY], bzh = k.u[U_BZ];
    const double vxh = k.u[U_RX] / roh;
    const double vyh = k.u[U_RY] / roh;
    const double vzh = k.u[U_RZ] / roh;
    const double vv = vxh * vxh + vyh * vyh + vzh * vzh;
    const double bb = bxh * bxh + byh * byh + bzh * bzh;
    const double prh = (gm - 1.0) * (eeh - 0.5 * roh * vv - pi8i * bb);
    const double exh = -vyh * bzh + vzh * byh;
    const double eyh = -vzh * bxh + vxh * bzh;
    const double ezh = -vxh * byh + vyh * bxh;
    const double ep = prh * gm / (gm - 1.0) + 0.5 * roh * vv;
    k.rox = roh * vxh;
    k.roy = roh * vyh;
    k.eex = ep * vxh + (bzh * eyh - byh * ezh) * pi4i;
    k.eey = ep * vyh + (bxh * ezh - bzh * exh) * pi4i;
    k.rxx = roh * (vxh * vxh) + prh + pi8i * (byh * byh + bzh * bzh - bxh * bxh);
    k.rxy = roh * vxh * vyh - pi4i * bxh * byh;
    k.ryx = roh * vyh * vxh - pi4i * byh * bxh;
    k.ryy = roh * (vyh * vyh) + prh + pi8i * (bxh * bxh + bzh * bzh - byh * byh);
    k.rzx = roh * vzh * vxh - pi4i * bzh * bxh;
    k.rzy = roh * vzh * vyh - pi4i * bzh * byh;
    k.nex = -exh;
    k.ey = eyh;
    k.ez = ezh;
}

// What an equation keeps of its cell values until its corner fluxes are
// there: the centred term of mlwhalf (mlwhalf.f:36-41) and the two terms of
// mlwartv (mlwartv.f:33-41)
struct Part {
    double du, ax, ay;
};
CANS_DEV void visc(const RowCoef &r, const Quad &u, double *pk, int q, Part &p) {
    const double dE = u.B - u.A, dW = shr1(dE), dN = u.C - u.A;
    p.ax = r.dt * (r.dxi * (r.qxe * dE - r.qxw * dW));
    p.ay = r.dt * (r.dyi * (r.qyn * dN - r.qys * pk[(K_DS + q) * WAVE]));
    pk[(K_DS + q) * WAVE] = dN;
}
// ro ee rx ry rz bz: an x flux f and a y flux g, w the slot of g
CANS_DEV double cells_xy(const RowCoef &r, const Quad &u, const Quad &f, const Quad &g, double dxim, double dyim,
                         double *pk, int q, int w, Part &p) {
    const double dfx = f.B - shr1(f.A);
    const double dgy = g.C - pk[(K_SY + w) * WAVE];
    pk[(K_SY + w) * WAVE] = g.A;
    p.du = 0.0;
    p.du = p.du - r.hdt * (r.hdxi * dfx) - r.hdt * (r.hdyi * dgy);
    visc(r, u, pk, q, p);
    return hu(u) - hx(f, dxim, r.dt) - hy(g, dyim, r.dt);
}
// the corner part (mlwfull.f:31-41), h and k the corner's x and y flux; wx,
// wy their slots
CANS_DEV double corner_dx(const RowCoef &r, double h, double *pk, int wx) {
    const double hN = h - shr1(h);
    const double d = r.dxi * (r.uy0 * pk[(K_DX + wx) * WAVE] + r.uy1 * hN);
    pk[(K_DX + wx) * WAVE] = hN;
    return d;
}
CANS_DEV double corner_dy(const RowCoef &r, double k, double *pk, int wy) {
    const double kE = k - pk[(K_KY + wy) * WAVE];
    pk[(K_KY + wy) * WAVE] = k;
    return r.dyi * (r.ux0 * shr1(kE) + r.ux1 * kE);
}
CANS_DEV double full_xy(const RowCoef &r, const Part &p, double h, double k, double *pk, int wx, int wy) {
    const double dfdx = corner_dx(r, h, pk, wx), dfdy = corner_dy(r, k, pk, wy);
    double du = p.du;
    du = du - r.hdt * dfdx - r.hdt * dfdy;
    du = du + p.ax + p.ay;
    return du;
}

// Primitive recovery (mlw_m3.f:340-374), the stores of cell (i, j) and of its
// images, and its cfl_m3 term.  With per_margin = m > 0 only the interior,
// [m+1, n-m] on both axes, stores: the fill replaces the rest.
template <class M, class P>
CANS_DEV void finish_row(const Mlw3Args &a, const M &map, const YMet<P> &y, const ColCtx &x, int j, const double *nu,
                         double az, bool do_cfl, double &dtmin_local) {
    const int ix = a.ix, jx = a.jx, mg = a.per_margin, i = x.i;
    const bool out = x.out && (mg == 0 || (j >= mg + 1 && j <= jx - mg));
    const bool edge = mg > 0 && (j <= 2 * mg + 1 || j >= jx - 2 * mg);   // rows that may have images
    const double gm = a.gm;
    const double ro = nu[U_RO], bx = nu[U_BX], by = nu[U_BY], bz = nu[U_BZ];
    const double vx = nu[U_RX] / ro;
    const double vy = nu[U_RY] / ro;
    const double vz = nu[U_RZ] / ro;
    const double vv = vx * vx + vy * vy + vz * vz;
    const double bb = bx * bx + by * by + bz * bz;
    const double pr = (gm - 1.0) * (nu[U_EE] - 0.5 * ro * vv - pi8i * bb);
    Faces faces{0xffu, {0u, 0u}};                                        // all BM_PER
    if constexpr (kMapped<M>) faces = map;
    if (do_cfl) {
        // v2 and b2 of cfl_m3 are vv and bb (the same sums, z components last);
        // the images' terms through the smallest spacing (cans_clock.hpp)
        const double dyg = edge ? images_min(faces.here(), 1, y.dy, j, jx, mg) : y.dy[j - 1];
        const double q = cfl2_term(a.safety, gm, ro, pr, vv, bb, fminF(x.dxg, dyg));
        dtmin_local = (out && q < dtmin_local) ? q : dtmin_local;
    }
    if (!out) return;
    const size_t rw = (size_t)(__builtin_amdgcn_readfirstlane(j) - 1) * (size_t)ix;
    unsigned bo = x.boff;
    asm volatile("" : "+v"(bo));
    st(a.out[0] + rw, bo, ro); st(a.out[1] + rw, bo, pr); st(a.out[2] + rw, bo, vx); st(a.out[3] + rw, bo, vy);
    st(a.out[4] + rw, bo, vz); st(a.out[5] + rw, bo, bx); st(a.out[6] + rw, bo, by); st(a.out[7] + rw, bo, bz);
    st(a.out[8] + rw, bo, az);
    if (!edge && !(mg > 0 && x.edge)) return;                            // uniform
    const Faces f = faces.here();
    const Images xi = images_of(f, 0, i, ix, mg), yj = images_of(f, 1, j, jx, mg);
    for (int b = -1; b < yj.count(); b++) {
        const int tj = b < 0 ? j : yj.at(b);
        const unsigned ny = b < 0 ? 0u : f.sign(1, b < yj.lo_n ? 0 : 1);
        for (int c = b < 0 ? 0 : -1; c < xi.count(); c++) {
            const int t = c < 0 ? i : xi.at(c);
            const unsigned ng = ny ^ (c < 0 ? 0u : f.sign(0, c < xi.lo_n ? 0 : 1));
            const size_t q = (size_t)(t - 1) + (size_t)ix * (size_t)(tj - 1);
            a.out[0][q] = ng & 1u ? -ro : ro; a.out[1][q] = ng & 2u ? -pr : pr;
            a.out[2][q] = ng & 4u ? -vx : vx; a.out[3][q] = ng & 8u ? -vy : vy;
            a.out[4][q] = ng & 16u ? -vz : vz; a.out[5][q] = ng & 32u ? -bx : bx;
            a.out[6][q] = ng & 64u ? -by : by; a.out[7][q] = ng & 128u ? -bz : bz;
            a.out[8][q] = ng & 256u ? -az : az;
        }
    }
}

// One output row: c the cell (i,j), R2 the cell (i,j+1) formed here, which
// the next row starts from; nxt the primitives of row j+1, replaced by those of
// row j+2; park the lane's LDS slots.
template <class M, class P>
CANS_DEV void row_step(const Mlw3Args &a, const M &map, const YMet<P> &y, const ColCtx &x, int j, double dt,
                       double z, bool do_cfl, const Cell &c, Cell &R2, Prim &nxt, double *park, double &dtmin_local) {
    j = __builtin_amdgcn_readfirstlane(j);
    // opaque, so that a row's parked values go through LDS and not through
    // registers to the next row
    unsigned po = 0;
    asm volatile("" : "+v"(po));
    double *pk = park + po;
    const double gm = a.gm;
    R2 = make_cell(nxt, gm);
    nxt = load_prim(a, x, j + 2);
    unsigned bo = x.boff;
    asm volatile("" : "+v"(bo));
    const double az = ld(row_of(a.in[8], a.ix, a.jx, j), bo);

    const double dyim = y.dim[j - 1], dxim = x.dxim;
    const double qxc = av_coef(x.qxs, shl1(c.vx), c.vx);
    const double qyc = av_coef(a.qav * y.dym[j - 1], R2.vy, c.vy);
    RowCoef r;
    r.hdt = 0.5 * dt;
    r.dt = dt;
    r.dxi = x.dxi;
    r.hdxi = 0.5 * x.dxi;
    r.dyi = y.di[j - 1];
    r.hdyi = 0.5 * r.dyi;
    r.ux0 = x.ux0; r.ux1 = x.ux1;
    r.uy0 = y.u0[j - 1]; r.uy1 = y.u1[j - 1];
    r.qxe = qxc * dxim;
    r.qxw = shr1(qxc) * x.dxim1;
    r.qyn = qyc * dyim;
    r.qys = pk[K_QY * WAVE] * y.dim[j - 2];
    pk[K_QY * WAVE] = qyc;

    // cell values
    Corner C;
    Part p[NU];
    const Quad qrx = quad(c.u[U_RX], R2.u[U_RX]), qry = quad(c.u[U_RY], R2.u[U_RY]);
    C.u[U_RO] = cells_xy(r, quad(c.u[U_RO], R2.u[U_RO]), qrx, qry, dxim, dyim, pk, U_RO, W_RO, p[U_RO]);
    C.u[U_RX] = cells_xy(r, qrx, quad(c.rxx, R2.rxx), quad(c.rxy, R2.rxy), dxim, dyim, pk, U_RX, W_RX, p[U_RX]);
    C.u[U_RY] = cells_xy(r, qry, quad(c.ryx, R2.ryx), quad(c.ryy, R2.ryy), dxim, dyim, pk, U_RY, W_RY, p[U_RY]);
    C.u[U_RZ] = cells_xy(r, quad(c.u[U_RZ], R2.u[U_RZ]), quad(c.rzx, R2.rzx), quad(c.rzy, R2.rzy), dxim, dyim, pk,
                         U_RZ, W_RZ, p[U_RZ]);
    C.u[U_EE] = cells_xy(r, quad(c.u[U_EE], R2.u[U_EE]), quad(c.eex, R2.eex), quad(c.eey, R2.eey), dxim, dyim, pk,
                         U_EE, W_EE, p[U_EE]);
    C.u[U_BZ] = cells_xy(r, quad(c.u[U_BZ], R2.u[U_BZ]), quad(c.ey, R2.ey), quad(c.nex, R2.nex), dxim, dyim, pk,
                         U_BZ, W_BZ, p[U_BZ]);
    const Quad qez = quad(c.ez, R2.ez);
    {   // bx: x flux 0, y flux ez
        const Quad u = quad(c.u[U_BX], R2.u[U_BX]);
        const double dgy = qez.C - pk[(K_SY + W_BX) * WAVE];
        pk[(K_SY + W_BX) * WAVE] = qez.A;
        p[U_BX].du = 0.0;
        p[U_BX].du = p[U_BX].du - z - r.hdt * (r.hdyi * dgy);
        visc(r, u, pk, U_BX, p[U_BX]);
        C.u[U_BX] = hu(u) - z - hy(qez, dyim, dt);
    }
    {   // by: x flux -ez (differences taken west - east, the same bits), y flux 0
        const Quad u = quad(c.u[U_BY], R2.u[U_BY]);
        p[U_BY].du = 0.0;
        p[U_BY].du = p[U_BY].du - r.hdt * (r.hdxi * (shr1(qez.A) - qez.B)) - z;
        visc(r, u, pk, U_BY, p[U_BY]);
        C.u[U_BY] = hu(u) - hx(Quad{-qez.A, -qez.B, -qez.C, -qez.D}, dxim, dt) - z;
    }
    // Az: mlwsrch.f:32-36 then mlwsrcf.f:33-40, source s = -ez
    double daz = 0.0;
    daz = daz + r.hdt * (-c.ez);

    corner_fluxes(C, gm);

    double nu[NU];
    nu[U_RO] = c.u[U_RO] + full_xy(r, p[U_RO], C.rox, C.roy, pk, W_RO, W_RO);
    nu[U_EE] = c.u[U_EE] + full_xy(r, p[U_EE], C.eex, C.eey, pk, W_EE, W_EE);
    nu[U_RX] = c.u[U_RX] + full_xy(r, p[U_RX], C.rxx, C.rxy, pk, W_RX, W_RX);
    nu[U_RY] = c.u[U_RY] + full_xy(r, p[U_RY], C.ryx, C.ryy, pk, W_RY, W_RY);
    nu[U_RZ] = c.u[U_RZ] + full_xy(r, p[U_RZ], C.rzx, C.rzy, pk, W_RZ, W_RZ);
    nu[U_BZ] = c.u[U_BZ] + full_xy(r, p[U_BZ], C.ey, C.nex, pk, W_BZ, W_BZ);
    const double ezW = shr1(C.ez);
    {
        const double dfdy = corner_dy(r, C.ez, pk, W_BX);
        double du = p[U_BX].du;
        du = du - z - r.hdt * dfdy;
        du = du + p[U_BX].ax + p[U_BX].ay;
        nu[U_BX] = c.u[U_BX] + du;
    }
    {
        const double hN = ezW - C.ez;
        const double dfdx = r.dxi * (r.uy0 * pk[(K_DX + W_BY) * WAVE] + r.uy1 * hN);
        pk[(K_DX + W_BY) * WAVE] = hN;
        double du = p[U_BY].du;
        du = du - r.hdt * dfdx - z;
        du = du + p[U_BY].ax + p[U_BY].ay;
        nu[U_BY] = c.u[U_BY] + du;
    }
    const double PN = x.ux0 * (-ezW) + x.ux1 * (-C.ez);
    const double sh = r.uy0 * pk[K_PS * WAVE] + r.uy1 * PN;
    pk[K_PS * WAVE] = PN;
    daz = daz + r.hdt * sh;

    finish_row(a, map, y, x, j, nu, az + daz, do_cfl, dtmin_local);
}

// One wave's strip of columns, output rows jb = 2+rowb*H .. min(jb+H-1, jx-1),
// after the cells of rows jb-1 and jb and the corner row jb-1.
template <class M, class P>
CANS_DEV void march_strip(const Mlw3Args &a, const M &map, const YMet<P> &y, int H, int strip, int rowb, double dt,
                          bool do_cfl, double *park, double &dtmin_local) {
    const int jx = a.jx;
    const int jb = 2 + rowb * H;
    const int je = min(jb + H - 1, jx - 1);
    __builtin_amdgcn_s_setprio(3);         // issue priority by progress, as cans_mlw2d.hip
    ColCtx x = column_of(a, map, strip);
    if constexpr (!kMapped<M>) x.edge = strip * COLS < 2 * a.per_margin + 1 || (strip + 1) * COLS + 1 >= a.ix - 2 * a.per_margin;
    const double z = dt * 0.0;

    Cell c0 = make_cell(load_prim(a, x, jb - 1), a.gm), c1 = make_cell(load_prim(a, x, jb), a.gm);
    Prim nxt = load_prim(a, x, jb + 1);
    {
        const Cell &A = c0, &N = c1;
        const double dxim = x.dxim, dyim = a.my.dim[jb - 2];
        const Quad rx = quad(A.u[U_RX], N.u[U_RX]), ry = quad(A.u[U_RY], N.u[U_RY]), ez = quad(A.ez, N.ez);
        Corner C;
        auto half = [&](double ua, double un, const Quad &f, const Quad &g) {
            return hu(quad(ua, un)) - hx(f, dxim, dt) - hy(g, dyim, dt);
        };
        C.u[U_RO] = half(A.u[U_RO], N.u[U_RO], rx, ry);
        C.u[U_EE] = half(A.u[U_EE], N.u[U_EE], quad(A.eex, N.eex), quad(A.eey, N.eey));
        C.u[U_RX] = half(A.u[U_RX], N.u[U_RX], quad(A.rxx, N.rxx), quad(A.rxy, N.rxy));
        C.u[U_RY] = half(A.u[U_RY], N.u[U_RY], quad(A.ryx, N.ryx), quad(A.ryy, N.ryy));
        C.u[U_RZ] = half(A.u[U_RZ], N.u[U_RZ], quad(A.rzx, N.rzx), quad(A.rzy, N.rzy));
        C.u[U_BZ] = half(A.u[U_BZ], N.u[U_BZ], quad(A.ey, N.ey), quad(A.nex, N.nex));
        C.u[U_BX] = hu(quad(A.u[U_BX], N.u[U_BX])) - z - hy(ez, dyim, dt);
        C.u[U_BY] = hu(quad(A.u[U_BY], N.u[U_BY])) - hx(Quad{-ez.A, -ez.B, -ez.C, -ez.D}, dxim, dt) - z;
        corner_fluxes(C, a.gm);
        const double ezW = shr1(C.ez);
        const double sy[7] = {A.u[U_RY], A.eey, A.rxy, A.ryy, A.rzy, A.ez, A.nex};
        const double ky[7] = {C.roy, C.eey, C.rxy, C.ryy, C.rzy, C.ez, C.nex};
        const double dX[7] = {C.rox - shr1(C.rox), C.eex - shr1(C.eex), C.rxx - shr1(C.rxx), C.ryx - shr1(C.ryx),
                              C.rzx - shr1(C.rzx), ezW - C.ez, C.ey - shr1(C.ey)};
#pragma unroll
        for (int q = 0; q < 7; q++) {
            park[(K_SY + q) * WAVE] = sy[q];
            park[(K_KY + q) * WAVE] = ky[q];
            park[(K_DX + q) * WAVE] = dX[q];
        }
#pragma unroll
        for (int q = 0; q < NU; q++) park[(K_DS + q) * WAVE] = N.u[q] - A.u[q];
        park[K_PS * WAVE] = x.ux0 * (-ezW) + x.ux1 * (-C.ez);
        park[K_QY * WAVE] = av_coef(a.qav * a.dym[jb - 2], N.vy, A.vy);
    }

    // two rows per trip, the cells changing places
    int j = jb;
    const int nr = je - jb + 1;
    for (; j + 1 <= je; j += 2) {
        const int q4 = (4 * (j - jb)) / nr;
        if (q4 == 1) __builtin_amdgcn_s_setprio(2);
        else if (q4 == 2) __builtin_amdgcn_s_setprio(1);
        else if (q4 >= 3) __builtin_amdgcn_s_setprio(0);
        row_step(a, map, y, x, j, dt, z, do_cfl, c1, c0, nxt, park, dtmin_local);
        row_step(a, map, y, x, j + 1, dt, z, do_cfl, c0, c1, nxt, park, dtmin_local);
    }
    if (j <= je) row_step(a, map, y, x, j, dt, z, do_cfl, c1, c0, nxt, park, dtmin_local);
}

template <class M>
__global__ __launch_bounds__(WAVE * WPB) __attribute__((amdgpu_waves_per_eu(2))) void mlw2d_m3_kernel(
    Mlw3Args a, M map, int H, const double *__restrict__ ydim, const double *__restrict__ ydi,
    const double *__restrict__ yu0, const double *__restrict__ yu1, const double *__restrict__ ydym,
    const double *__restrict__ ydy) {
    const YMet<const double *> y{ydim, ydi, yu0, yu1, ydym, ydy};
    __shared__ double red[WPB];
    __shared__ double park[WPB][NK][WAVE];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nstrip = (a.ix - 2 + COLS - 1) / COLS;
    const int nrowb = (a.jx - 2 + H - 1) / H;
    const int nblocks = (nstrip * nrowb + WPB - 1) / WPB;
    const int unit = xcd_remap(blockIdx.x, nblocks) * WPB + wv;
    double dt = a.dt;
    if (a.clk) {   // per_margin > 0: the kernel advances the clock, else a clock kernel did
        const StepCtl c = clock_use(a.clk, a.step, a.per_margin == 0, blockIdx.x == 0 && threadIdx.x == 0);
        if (!c.run) return;                // uniform across the launch
        dt = c.dt;
    }
    const bool do_cfl = a.clk && a.safety > 0.0;
    double dtmin_local = kR4_1e20;
    if (unit < nstrip * nrowb)
        march_strip(a, map, y, H, unit % nstrip, unit / nstrip, dt, do_cfl, &park[wv][0][threadIdx.x & (WAVE - 1)],
                    dtmin_local);
    if (do_cfl) block_min_to_global(dtmin_local, red, &a.clk->dtkey[(a.step + 1) % 3]);
}

}  // namespace

hipError_t launch_mlw2d_m3(const Mlw3Args &a, hipStream_t s, const BndMap *map) {
    if (a.ix < 3 || a.jx < 3) return hipSuccess;
    const int h = pick_rows(a.ix, a.jx);
    const int nstrip = (a.ix - 2 + COLS - 1) / COLS;
    const int nrowb = (a.jx - 2 + h - 1) / h;
    const int nblocks = (nstrip * nrowb + WPB - 1) / WPB;
    if (map)
        hipLaunchKernelGGL((mlw2d_m3_kernel<Faces>), dim3(nblocks), dim3(WAVE * WPB), 0, s, a, pack_faces(*map), h,
                           a.my.dim, a.my.di, a.my.u0, a.my.u1, a.dym, a.dy);
    else
        hipLaunchKernelGGL((mlw2d_m3_kernel<PerBox>), dim3(nblocks), dim3(WAVE * WPB), 0, s, a, PerBox{}, h, a.my.dim,
                           a.my.di, a.my.u0, a.my.u1, a.dym, a.dy);
    return hipGetLastError();
}

}  // namespace cans

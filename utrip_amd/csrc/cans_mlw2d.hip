// cans_mlw2d.hip -- fused 2D modified Lax-Wendroff MHD step (gfx950).
//
// One launch does the whole of cans2d/hdmlw/mlw_m.f:2-324 (mlwhalf, mlwsrch,
// mlwfull, mlwsrcf, mlwartv, update, primitive recovery), and optionally the
// periodic ghost fill of cans2d/bc/bdper{x,y}.f and the CFL reduction of
// cans2d/common/cfl_m.f for the next step.  State is structure-of-arrays
// FP64, column-major (ix,jx) as the reference holds it.
//
// Mapping: one wavefront owns a strip of 64 columns (62 output columns and
// one halo column each side) and marches along y over H output rows.  The
// stencil rows live in registers; x neighbours come from the adjacent lanes
// through DPP wave shifts (v_mov_b32_dpp wave_shl:1 / wave_shr:1), so there is
// no LDS traffic and no barrier, and each field is read once per strip and
// row with coalesced 512-byte wave loads.  The carried row state is kept to
// what the next row cannot re-derive by a lane shift (the east cell is
// shifted again rather than carried), so that a wave fits in 256 VGPRs and
// two waves share each SIMD: the FP64 chains of one hide the latency of the
// other's.
//
// Per output row j a lane forms the cell state of row j+1 (mlw_m.f:101-176),
// the corner half step (i,j) between rows j and j+1 (mlwhalf.f:45-52,
// mlw_m.f:189-262), and the update of cell (i,j).  Differences that the
// reference forms for two neighbouring cells are the same IEEE operation on
// the same operands -- e.g. (u(i+1)-u(i)) is uE-uc of cell i and uc-uW of
// cell i+1 (mlwartv.f:33-41), the corner-flux difference of corner row j is
// the north difference of row j and the south difference of row j+1
// (mlwfull.f:31-41) -- so each is computed once and handed to the neighbour
// by a lane shift or carried to the next row.  Every value is formed by the
// reference's expression in the reference's order, so the results are
// bit-identical to it and independent of the strip decomposition.
#include "cans_common.hpp"
#include "cans_clock.hpp"
#include "cans_kernels.hpp"
#include "cans_march2d.hpp"
#include "cans_wave.hpp"

namespace cans {
using namespace march2d;
namespace {

constexpr int kOccBatch = 2;                 // waves per SIMD of the batched kernel (the strip's registers)
// u: ro ee rx ry bx by (the six conserved variables, mlw_m.f:101-112)
enum { U_RO, U_EE, U_RX, U_RY, U_BX, U_BY, NU };

struct Prim {
    double ro, pr, vx, vy, bx, by;
};

// Conserved variables and cell-centred fluxes of one cell (mlw_m.f:101-176).
// x fluxes of the six equations: rx, eex, rxx, ryx, 0, -ez
// y fluxes:                      ry, eey, rxy, ryy, ez, 0
struct Cell {
    double u[NU];
    double eex, eey, rxx, rxy, ryx, ryy, ez;
    double vx, vy;
};

// The part of the east neighbour a cell needs (no vy).
struct CellE {
    double u[NU];
    double eex, eey, rxx, rxy, ryx, ryy, ez;
    double vx;
};

struct Corner {
    double rox, roy, eex, eey, rxx, rxy, ryx, ryy, ez;
};

// Row state carried from output row j-1 to output row j.
struct RowState {
    Cell c;          // cell (i, j)
    double sy[5];    // y fluxes ry eey rxy ryy ez of cell (i, j-1)
    double dS[NU];   // u(i,j) - u(i,j-1)               (= uc - uS of row j)
    double qys;      // AV coefficient of face j-1/2
    double ky[5];    // y fluxes roy eey rxy ryy ez of corner (i, j-1)
    double dXS[5];   // corner x-flux differences of corner row j-1
    double PS;       // ux0*(-ezh(i-1,j-1)) + ux1*(-ezh(i,j-1))
    Prim nxt;        // primitives of cell (i, j+1), loaded
    double az;       // az of cell (i, j), loaded
    double pro, pee, prx, pry, pbx, pby, paz;   // updated cell (i, j)
};

CANS_DEV Prim load_prim(const Mlw2dArgs &a, const ColCtx &x, int j) {
    const size_t r = row_of(a.ro, a.ix, a.jx, j) - a.ro;
    // Loads as scalar row base + 32-bit lane offset; the empty asm keeps the
    // compiler from hoisting six 64-bit per-lane field pointers into VGPRs.
    unsigned bo = x.boff;
    asm volatile("" : "+v"(bo));
    Prim p;
    p.ro = ld(a.ro + r, bo); p.pr = ld(a.pr + r, bo); p.vx = ld(a.vx + r, bo);
    p.vy = ld(a.vy + r, bo); p.bx = ld(a.bx + r, bo); p.by = ld(a.by + r, bo);
    return p;
}

CANS_DEV double load_az(const Mlw2dArgs &a, const ColCtx &x, int j) {
    unsigned bo = x.boff;
    asm volatile("" : "+v"(bo));
    return ld(row_of(a.az, a.ix, a.jx, j), bo);
}

// mlw_m.f:101-176 for one cell
CANS_DEV Cell make_cell(const Prim &p, double gm) {
    Cell c;
    const double ro = p.ro, pr = p.pr, vx = p.vx, vy = p.vy, bx = p.bx, by = p.by;
    const double vv = vx * vx + vy * vy;
    const double bb = bx * bx + by * by;
    const double ez = -vx * by + vy * bx;
    const double ep = pr * gm / (gm - 1.0) + 0.5 * ro * vv;
    c.u[U_RO] = ro;
    c.u[U_EE] = pr / (gm - 1.0) + 0.5 * ro * vv + pi8i * bb;
    c.u[U_RX] = ro * vx;
    c.u[U_RY] = ro * vy;
    c.u[U_BX] = bx;
    c.u[U_BY] = by;
    c.eex = ep * vx - by * ez * pi4i;
    c.eey = ep * vy + bx * ez * pi4i;
    c.rxx = ro * (vx * vx) + pr + pi8i * (by * by - bx * bx);
    c.rxy = ro * vx * vy - pi4i * bx * by;
    c.ryx = ro * vy * vx - pi4i * by * bx;
    c.ryy = ro * (vy * vy) + pr + pi8i * (bx * bx - by * by);
    c.ez = ez;
    c.vx = vx;
    c.vy = vy;
    return c;
}

CANS_DEV CellE shl_cell(const Cell &c) {
    CellE r;
#pragma unroll
    for (int q = 0; q < NU; q++) r.u[q] = shl1(c.u[q]);
    r.eex = shl1(c.eex); r.eey = shl1(c.eey); r.rxx = shl1(c.rxx); r.rxy = shl1(c.rxy);
    r.ryx = shl1(c.ryx); r.ryy = shl1(c.ryy); r.ez = shl1(c.ez); r.vx = shl1(c.vx);
    return r;
}

// corner between columns i,i+1 and rows j,j+1 (mlwhalf.f:45-52, mlw_m.f:189-262)
template <class CA, class CB>
CANS_DEV Corner make_corner(const CA &A, const CB &B, const CA &C, const CB &D, double dxim, double dyim, double dt,
                            double gm) {
    const double roh = half1(A.u[U_RO], B.u[U_RO], C.u[U_RO], D.u[U_RO], A.u[U_RX], B.u[U_RX], C.u[U_RX],
                             D.u[U_RX], A.u[U_RY], B.u[U_RY], C.u[U_RY], D.u[U_RY], dxim, dyim, dt);
    const double eeh = half1(A.u[U_EE], B.u[U_EE], C.u[U_EE], D.u[U_EE], A.eex, B.eex, C.eex, D.eex, A.eey, B.eey,
                             C.eey, D.eey, dxim, dyim, dt);
    const double rxh = half1(A.u[U_RX], B.u[U_RX], C.u[U_RX], D.u[U_RX], A.rxx, B.rxx, C.rxx, D.rxx, A.rxy, B.rxy,
                             C.rxy, D.rxy, dxim, dyim, dt);
    const double ryh = half1(A.u[U_RY], B.u[U_RY], C.u[U_RY], D.u[U_RY], A.ryx, B.ryx, C.ryx, D.ryx, A.ryy, B.ryy,
                             C.ryy, D.ryy, dxim, dyim, dt);
    const double bxh = half1_y(A.u[U_BX], B.u[U_BX], C.u[U_BX], D.u[U_BX], A.ez, B.ez, C.ez, D.ez, dyim, dt);
    const double byh = half1_x(A.u[U_BY], B.u[U_BY], C.u[U_BY], D.u[U_BY], -A.ez, -B.ez, -C.ez, -D.ez, dxim, dt);
    const double vxh = rxh / roh;
    const double vyh = ryh / roh;
    const double vv = vxh * vxh + vyh * vyh;
    const double bb = bxh * bxh + byh * byh;
    const double prh = (gm - 1.0) * (eeh - 0.5 * roh * vv - pi8i * bb);
    const double ezh = -vxh * byh + vyh * bxh;
    const double ep = prh * gm / (gm - 1.0) + 0.5 * roh * vv;
    Corner k;
    k.rox = roh * vxh;
    k.roy = roh * vyh;
    k.eex = ep * vxh - byh * ezh * pi4i;
    k.eey = ep * vyh + bxh * ezh * pi4i;
    k.rxx = roh * (vxh * vxh) + prh + pi8i * (byh * byh - bxh * bxh);
    k.rxy = roh * vxh * vyh - pi4i * bxh * byh;
    k.ryx = roh * vyh * vxh - pi4i * byh * bxh;
    k.ryy = roh * (vyh * vyh) + prh + pi8i * (bxh * bxh - byh * byh);
    k.ez = ezh;
    return k;
}

// One equation with both an x and a y flux (ro ee rx ry).  f*: cell x flux,
// g*: cell y flux, h*: corner x flux, k*: corner y flux.  The differences
// handed on: hN (south difference of the next row), kE (shifted to the east
// neighbour as its kW), dN (the next row's dS).
CANS_DEV double eq_xy(const RowCoef &r, double fE, double fC, double gN, double gS, double hC, double hS, double kC,
                      double kS, double uE, double uc, double uN, double dS, double &hN, double &dN) {
    const double dfx = fE - shr1(fC);
    const double dgy = gN - gS;
    hN = hC - shr1(hC);
    const double kE = kC - kS;
    const double kW = shr1(kE);
    const double dE = uE - uc;
    const double dW = shr1(dE);
    dN = uN - uc;
    return du1(r, dfx, dgy, hS, hN, kW, kE, dE, dW, dN, dS);
}

// Primitive recovery (mlw_m.f:299-321), the CFL term of the new state
// (cans2d/common/cfl_m.f:46-55) and the stores of the updated cell (i, j),
// with its periodic ghost images.  When the kernel writes the ghost images
// (per_margin = m > 0) only interior cells, i in [m+1, ix-m] and j in
// [m+1, jx-m], store and enter the CFL: the reference's bdperx/bdpery
// overwrite what mlw_m computed in the ghost cells 2..m and ix-m+1..ix-1
// with interior images.
template <class M, class P>
CANS_DEV void finish_row(const Mlw2dArgs &a, const M &map, const YMet<P> &y, const ColCtx &x, int j, const RowState &s,
                         bool do_cfl, double &dtmin_local) {
    const int mgj = a.per_margin;
    const bool out = x.out && (mgj == 0 || (j >= mgj + 1 && j <= a.jx - mgj));   // uniform in j
    const double gm = a.gm;
    const double ro = s.pro, ee = s.pee, rx = s.prx, ry = s.pry, bx = s.pbx, by = s.pby, az = s.paz;
    const double vx = rx / ro;
    const double vy = ry / ro;
    const double vv = vx * vx + vy * vy;
    const double bb = bx * bx + by * by;
    const double pr = (gm - 1.0) * (ee - 0.5 * ro * vv - pi8i * bb);
    double sq = 0.0;
    if (do_cfl) {
        const double b2 = bx * bx + by * by;
        const double ca2 = b2 * pi4i / ro;
        const double cs2 = gm * pr / ro;
        const double v2 = vx * vx + vy * vy;
        sq = __builtin_sqrt(v2 + cs2 + ca2);
        // The reference's cfl_m also visits the periodic ghost images of
        // this cell, which hold the same state: their terms are
        // safety*(min(dx(gi), dy(gj))/sq) over the images (gi, gj).  For
        // sq >= 0, m -> safety*(m/sq) is monotone non-decreasing in IEEE
        // arithmetic (a NaN sq gives NaN terms that never win either way), so
        // the smallest of those terms is safety*(min(min dx, min dy)/sq) bit
        // for bit: one division per cell and no per-image metric loads.
        const int mg = a.per_margin, jx = a.jx;
        double dyg = y.dy[j - 1];
        if constexpr (kMapped<M>) {
            if (j <= 2 * mg + 1 || j >= jx - 2 * mg) dyg = images_min(map.here(), 1, y.dy, j, jx, mg);
        } else {
            if (mg > 0 && j >= jx - 2 * mg + 1) dyg = fminF(dyg, y.dy[j - (jx - 2 * mg) - 1]);
            if (mg > 0 && j <= 2 * mg) dyg = fminF(dyg, y.dy[j + (jx - 2 * mg) - 1]);
        }
        const double dtq = a.safety * (fminF(x.dxg, dyg) / sq);
        dtmin_local = (out && dtq < dtmin_local) ? dtq : dtmin_local;
    }
    if (out) {
        const int ix = a.ix, jx = a.jx;
        // Stores as scalar row address + 32-bit lane offset.  The empty asm
        // makes the offset opaque so that the compiler does not hoist seven
        // 64-bit per-lane field pointers out of the loop into registers.
        const size_t rw = (size_t)(__builtin_amdgcn_readfirstlane(j) - 1) * (size_t)ix;
        unsigned bo = x.boff;
        asm volatile("" : "+v"(bo));
        st(a.ro_o + rw, bo, ro); st(a.pr_o + rw, bo, pr); st(a.vx_o + rw, bo, vx);
        st(a.vy_o + rw, bo, vy); st(a.bx_o + rw, bo, bx); st(a.by_o + rw, bo, by);
        st(a.az_o + rw, bo, az);
        // In a periodic box also the ghost images: after bdperx then
        // bdpery, ghost (gi,gj) holds interior (src_x(gi), src_y(gj)); with a
        // map likewise, each field times the signs of the faces.
        const int mg = a.per_margin;   // the host checks ix-2m >= m and jx-2m >= m (bnd_map for a map)
        const int i = x.i;
        if constexpr (kMapped<M>) {
            if (x.edge || j <= 2 * mg + 1 || j >= jx - 2 * mg) {   // uniform
                const Faces map_ = map.here();
                const Images xi = images_of(map_, 0, i, ix, mg), yj = images_of(map_, 1, j, jx, mg);
                for (int b = -1; b < yj.count(); b++) {
                    const int tj = b < 0 ? j : yj.at(b);
                    const unsigned ny = b < 0 ? 0u : map_.sign(1, b < yj.lo_n ? 0 : 1);
                    for (int c = b < 0 ? 0 : -1; c < xi.count(); c++) {
                        const int t = c < 0 ? i : xi.at(c);
                        const unsigned ng = ny ^ (c < 0 ? 0u : map_.sign(0, c < xi.lo_n ? 0 : 1));
                        const size_t q = (size_t)(t - 1) + (size_t)ix * (size_t)(tj - 1);
                        a.ro_o[q] = ng & 1u ? -ro : ro; a.pr_o[q] = ng & 2u ? -pr : pr;
                        a.vx_o[q] = ng & 4u ? -vx : vx; a.vy_o[q] = ng & 8u ? -vy : vy;
                        a.bx_o[q] = ng & 16u ? -bx : bx; a.by_o[q] = ng & 32u ? -by : by;
                        a.az_o[q] = ng & 64u ? -az : az;
                    }
                }
            }
        } else if (mg > 0 && (i >= ix - 2 * mg + 1 || i <= 2 * mg || j >= jx - 2 * mg + 1 || j <= 2 * mg)) {
            int xi[3] = {i, 0, 0}, yj[3] = {j, 0, 0};
            int nxi = 1, nyj = 1;
            if (i >= ix - 2 * mg + 1) xi[nxi++] = i - (ix - 2 * mg);   // low ghost  <- high interior
            if (i <= 2 * mg) xi[nxi++] = i + (ix - 2 * mg);            // high ghost <- low interior
            if (j >= jx - 2 * mg + 1) yj[nyj++] = j - (jx - 2 * mg);
            if (j <= 2 * mg) yj[nyj++] = j + (jx - 2 * mg);
            for (int b = 0; b < nyj; b++) {
                for (int c = 0; c < nxi; c++) {
                    if (b == 0 && c == 0) continue;
                    const size_t q = (size_t)(xi[c] - 1) + (size_t)ix * (size_t)(yj[b] - 1);
                    a.ro_o[q] = ro; a.pr_o[q] = pr; a.vx_o[q] = vx; a.vy_o[q] = vy;
                    a.bx_o[q] = bx; a.by_o[q] = by; a.az_o[q] = az;
                }
            }
        }
    }
}

// One output row j: s holds the state entering row j, o receives the state
// entering row j+1.  Everything but the stores runs on all 64 lanes (the
// lane shifts need every lane's operands).
template <class M, class P>
CANS_DEV void row_step(const Mlw2dArgs &a, const M &map, const YMet<P> &y, const ColCtx &x, int j, double dt,
                       bool do_cfl, const RowState &s, RowState &o, double &dtmin_local) {
    j = __builtin_amdgcn_readfirstlane(j);   // wave-uniform: SGPR row bases and scalar loads
    const double gm = a.gm;
    // prefetch the row after next and the az of the next row
    o.nxt = load_prim(a, x, j + 2);
    o.az = load_az(a, x, j + 1);

    const double dyim = y.dim[j - 1];
    const CellE E = shl_cell(s.c);                 // cell (i+1, j)
    const Cell R2 = make_cell(s.nxt, gm);          // cell (i, j+1)
    const CellE R2p = shl_cell(R2);                // cell (i+1, j+1)
    const Corner C = make_corner(s.c, E, R2, R2p, x.dxim, dyim, dt, gm);

    const double qxc = av_coef(x.qxs, E.vx, s.c.vx);
    const double qyc = av_coef(a.qav * y.dym[j - 1], R2.vy, s.c.vy);
    RowCoef r;
    r.hdt = 0.5 * dt;
    r.dt = dt;
    r.dxi = x.dxi;
    r.hdxi = 0.5 * x.dxi;
    r.dyi = y.di[j - 1];
    r.hdyi = 0.5 * r.dyi;
    r.ux0 = x.ux0; r.ux1 = x.ux1;
    r.uy0 = y.u0[j - 1]; r.uy1 = y.u1[j - 1];
    r.qxe = qxc * x.dxim;
    r.qxw = shr1(qxc) * x.dxim1;
    r.qyn = qyc * dyim;
    r.qys = s.qys * y.dim[j - 2];

    double du[NU];
    du[U_RO] = eq_xy(r, E.u[U_RX], s.c.u[U_RX], R2.u[U_RY], s.sy[0], C.rox, s.dXS[0], C.roy, s.ky[0],
                     E.u[U_RO], s.c.u[U_RO], R2.u[U_RO], s.dS[U_RO], o.dXS[0], o.dS[U_RO]);
    du[U_EE] = eq_xy(r, E.eex, s.c.eex, R2.eey, s.sy[1], C.eex, s.dXS[1], C.eey, s.ky[1], E.u[U_EE],
                     s.c.u[U_EE], R2.u[U_EE], s.dS[U_EE], o.dXS[1], o.dS[U_EE]);
    du[U_RX] = eq_xy(r, E.rxx, s.c.rxx, R2.rxy, s.sy[2], C.rxx, s.dXS[2], C.rxy, s.ky[2], E.u[U_RX],
                     s.c.u[U_RX], R2.u[U_RX], s.dS[U_RX], o.dXS[2], o.dS[U_RX]);
    du[U_RY] = eq_xy(r, E.ryx, s.c.ryx, R2.ryy, s.sy[3], C.ryx, s.dXS[3], C.ryy, s.ky[3], E.u[U_RY],
                     s.c.u[U_RY], R2.u[U_RY], s.dS[U_RY], o.dXS[3], o.dS[U_RY]);
    const double ezW = shr1(C.ez);                 // ezh(i-1, j)
    {   // bx: x flux 0, y flux ez
        const double kE = C.ez - s.ky[4];
        const double dE = E.u[U_BX] - s.c.u[U_BX];
        const double dN = R2.u[U_BX] - s.c.u[U_BX];
        du[U_BX] = du1_y(r, R2.ez - s.sy[4], shr1(kE), kE, dE, shr1(dE), dN, s.dS[U_BX]);
        o.dS[U_BX] = dN;
    }
    {   // by: x flux -ez, y flux 0.  (-a)-(-b) is b-a bit for bit (signed
        // zeros included), so the x differences are taken as west - east.
        const double hN = ezW - C.ez;
        const double dE = E.u[U_BY] - s.c.u[U_BY];
        const double dN = R2.u[U_BY] - s.c.u[U_BY];
        du[U_BY] = du1_x(r, shr1(s.c.ez) - E.ez, s.dXS[4], hN, dE, shr1(dE), dN, s.dS[U_BY]);
        o.dXS[4] = hN;
        o.dS[U_BY] = dN;
    }
    // Az: mlwsrch.f:32-36 then mlwsrcf.f:33-40, source s = -ez
    const double PN = x.ux0 * (-ezW) + x.ux1 * (-C.ez);
    double daz = 0.0;
    daz = daz + r.hdt * (-s.c.ez);
    const double sh = r.uy0 * s.PS + r.uy1 * PN;
    daz = daz + r.hdt * sh;
    // update (mlw_m.f:299-304)
    o.pro = s.c.u[U_RO] + du[U_RO];
    o.pee = s.c.u[U_EE] + du[U_EE];
    o.prx = s.c.u[U_RX] + du[U_RX];
    o.pry = s.c.u[U_RY] + du[U_RY];
    o.pbx = s.c.u[U_BX] + du[U_BX];
    o.pby = s.c.u[U_BY] + du[U_BY];
    o.paz = s.az + daz;

    // state entering row j+1
    o.c = R2;
    o.sy[0] = s.c.u[U_RY]; o.sy[1] = s.c.eey; o.sy[2] = s.c.rxy; o.sy[3] = s.c.ryy; o.sy[4] = s.c.ez;
    o.qys = qyc;
    o.ky[0] = C.roy; o.ky[1] = C.eey; o.ky[2] = C.rxy; o.ky[3] = C.ryy; o.ky[4] = C.ez;
    o.PS = PN;

    finish_row(a, map, y, x, j, o, do_cfl, dtmin_local);
}

// One wave's strip: columns 1+strip*COLS .. (lane 0 the west halo), output
// rows jb = 2+rowb*H .. min(jb+H-1, jx-1), marched in y (prologue: the cells
// of rows jb-1 and jb and the corner row jb-1).
template <class M, class P>
CANS_DEV void march_strip(const Mlw2dArgs &a, const M &map, const YMet<P> &y, int H, int strip, int rowb, double dt,
                          bool do_cfl, double &dtmin_local) {
    const int jx = a.jx;
    const int jb = 2 + rowb * H;
    const int je = min(jb + H - 1, jx - 1);
    // Issue priority by progress: two waves share a SIMD, and with equal
    // priorities the older one issues first, finishes early and leaves the
    // younger one to end its rows alone, with its FP64 latencies exposed.  A
    // wave starts at priority 3 and steps down by one per quarter of its
    // rows, so the one further behind issues first and the pair ends
    // together (1024^2 step 38.0 -> 36.1 us, 4096^2 497 -> 488 us).
    __builtin_amdgcn_s_setprio(3);
    const ColCtx x = column_of(a, map, strip);

    // prologue: cells of rows jb-1 and jb, corner row jb-1
    const Cell R0 = make_cell(load_prim(a, x, jb - 1), a.gm);
    RowState s0, s1;
    s0.c = make_cell(load_prim(a, x, jb), a.gm);
    const CellE s0e = shl_cell(s0.c);
    s0.nxt = load_prim(a, x, jb + 1);
    s0.az = load_az(a, x, jb);
    const CellE R0p = shl_cell(R0);
    const Corner Cm = make_corner(R0, R0p, s0.c, s0e, x.dxim, a.my.dim[jb - 2], dt, a.gm);
    const double ezW = shr1(Cm.ez);
    s0.dXS[0] = Cm.rox - shr1(Cm.rox);
    s0.dXS[1] = Cm.eex - shr1(Cm.eex);
    s0.dXS[2] = Cm.rxx - shr1(Cm.rxx);
    s0.dXS[3] = Cm.ryx - shr1(Cm.ryx);
    s0.dXS[4] = ezW - Cm.ez;
    s0.PS = x.ux0 * (-ezW) + x.ux1 * (-Cm.ez);
    s0.ky[0] = Cm.roy; s0.ky[1] = Cm.eey; s0.ky[2] = Cm.rxy; s0.ky[3] = Cm.ryy; s0.ky[4] = Cm.ez;
    s0.sy[0] = R0.u[U_RY]; s0.sy[1] = R0.eey; s0.sy[2] = R0.rxy; s0.sy[3] = R0.ryy; s0.sy[4] = R0.ez;
#pragma unroll
    for (int q = 0; q < NU; q++) s0.dS[q] = s0.c.u[q] - R0.u[q];
    s0.qys = av_coef(a.qav * a.dym[jb - 2], s0.c.vy, R0.vy);

    // two rows per trip so that the carried state ping-pongs between
    // s0 and s1 instead of being copied
    int j = jb;
    const int nr = je - jb + 1;
    for (; j + 1 <= je; j += 2) {
        const int q4 = (4 * (j - jb)) / nr;   // quarters of the rows done
        if (q4 == 1) __builtin_amdgcn_s_setprio(2);
        else if (q4 == 2) __builtin_amdgcn_s_setprio(1);
        else if (q4 >= 3) __builtin_amdgcn_s_setprio(0);
        row_step(a, map, y, x, j, dt, do_cfl, s0, s1, dtmin_local);
        row_step(a, map, y, x, j + 1, dt, do_cfl, s1, s0, dtmin_local);
    }
    if (j <= je) row_step(a, map, y, x, j, dt, do_cfl, s0, s1, dtmin_local);
}

// The y metric arrays come as separate non-aliased arguments (the same
// pointers as a.my, a.dym, a.dy) so that their per-row uniform loads go
// through the scalar cache.
template <int OCC, class M>
__global__ __launch_bounds__(WAVE * WPB) __attribute__((amdgpu_waves_per_eu(OCC))) void mlw2d_kernel(
    Mlw2dArgs a, M map, int H, const double *__restrict__ ydim, const double *__restrict__ ydi,
    const double *__restrict__ yu0, const double *__restrict__ yu1, const double *__restrict__ ydym,
    const double *__restrict__ ydy) {
    const YMet<const double *> y{ydim, ydi, yu0, yu1, ydym, ydy};
    __shared__ double red[WPB];
    const int ix = a.ix, jx = a.jx;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nstrip = (ix - 2 + COLS - 1) / COLS;
    const int nrowb = (jx - 2 + H - 1) / H;
    const int nblocks = (nstrip * nrowb + WPB - 1) / WPB;
    const int unit = xcd_remap(blockIdx.x, nblocks) * WPB + wv;

    double dt = a.dt;
    bool run = true;
    if (a.clk) {
        StepCtl c = clock_use(a.clk, a.step, a.peek != 0, blockIdx.x == 0 && threadIdx.x == 0);
        run = c.run;
        dt = c.dt;
    }
    if (!run) return;                          // uniform across the launch
    if (a.dt_log && blockIdx.x == 0 && threadIdx.x == 0) a.dt_log[a.step] = dt;
    const bool do_cfl = a.clk && a.safety > 0.0;
    double dtmin_local = kR4_1e20;

    if (unit < nstrip * nrowb) march_strip(a, map, y, H, unit % nstrip, unit / nstrip, dt, do_cfl, dtmin_local);
    if (do_cfl) block_min_to_global(dtmin_local, red, &a.clk->dtkey[(a.step + 1) % 3]);
}

// ---------------------------------------------------------------- batched runs
// Many independent periodic 2D runs, each running the cans2d main loop
// (cans2d/md_mhdshktb/hdmlw/main.f:150-206 with bdperx/bdpery):
//     ns=ns+1; cfl_m; stop on merr; t=t+dt; mlw_m; bdperx; bdpery;
//     repeat while ns < nstop and t < tend
// to its own end, in one persistent kernel.  A step's work is its strips'
// units (march_strip: H rows of 62 columns, with the ghost images and the
// next step's cfl term), a wave a unit.
//
// A workgroup takes runs from a list, costliest first.  A small run (under
// kShareRounds rounds of units on the workgroup's waves) it advances by
// itself, a step a turn; its only synchronisation is the workgroup's.  The
// steps of a larger run are shared: whoever started the run, or finished the
// last unit of its step, puts the next step into the queue of its group of
// workgroups (those of one XCD, so that a run's state stays in one L2; runs
// are dealt to the groups in turn), and workgroups take NW units at a time
// from there, or from another group's when theirs has none, before anything
// else.  One workgroup per run left the card to the longest runs: 192 runs of
// 32..256 cells a side took 46.5 ms, the time of the costliest one on its CU.
//
// Nothing waits for a workgroup that may not be resident: a unit in a queue
// is ready to run, units are taken only by running workgroups, and the one
// that finishes a step's last unit queues the next.  A workgroup with
// nothing to do polls until there is no shared run left (`active`, raised
// before a run is taken from the list), which running workgroups bring about.  (The waiting inside a push is for an
// earlier push of the group to be published, a few instructions of a running
// wave.)
//
// Visibility: a wave waits for its stores (vmcnt 0) before the workgroup
// barrier, wave 0 then adds its units to the step's `done` count with
// agent-scope release; the last to add acquires, pushes with release (the
// word, then the tail), and who takes units acquires before its waves load.
enum { B2_UNITS, B2_OWN, B2_START, B2_IDLE, B2_EXIT };
// A run is shared from this many rounds of its workgroup's waves: at one round
// the queue costs more than it spreads (1000 runs of 16..64 cells a side 3.0
// against 1.1 ms), from two on it pays (192 runs of 32..256: 8.6 ms at two,
// 10.9 at three, 15.9 at six; 1024 such runs 37 ms, 71.3 unshared).
constexpr int kShareRounds = 2;
constexpr int kShareRuns = 1 << 24;        // run numbers fit a queue word
constexpr int kShareUnits = 1 << 15;       // units of a step fit a word

CANS_DEV unsigned long long ald(const unsigned long long *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
CANS_DEV unsigned ald(const unsigned *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
CANS_DEV int ald(const int *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <class T> CANS_DEV void ast(T *p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// one lane's atomic add, its old value in every lane
CANS_DEV unsigned add1(unsigned *p, unsigned v) {
    unsigned r = 0;
    if ((threadIdx.x & 63) == 0) r = __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return (unsigned)uni((int)r);
}
CANS_DEV unsigned long long add1(unsigned long long *p, unsigned long long v) {
    unsigned long long r = 0;
    if ((threadIdx.x & 63) == 0) r = __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return (unsigned long long)uni((long long)r);
}

// The rows per unit and the units of a run of ix x jx cells: the fewest
// rounds of NW units, a unit's prologue counted as 1.5 rows and its share of
// the round's synchronisation as 2.5.
struct B2Cut {
    int H, nstrip, nunit;
};
CANS_DEV B2Cut batch2d_cut(int ix, int jx, int NW) {
    B2Cut c{8, (ix - 2 + COLS - 1) / COLS, 0};
    double cost = 1e300;
    for (int h = 4; h <= 20; h++) {
        const int units = c.nstrip * ((jx - 2 + h - 1) / h);
        const double q = (double)((units + NW - 1) / NW) * (h + 4.0);
        if (q < cost) { cost = q; c.H = h; }
    }
    for (;; c.H *= 2) {
        c.nunit = c.nstrip * ((jx - 2 + c.H - 1) / c.H);
        if (c.nunit <= kShareUnits || c.H >= jx) break;
    }
    return c;
}

// The queue of a group: words (run, units, lap, next ticket) in a ring; [head,
// tail) are published, resv counts the reserved.  The lap of the ring (from 1,
// mod 64; an empty slot holds 0) says which of a slot's words one is: head and
// tail are read relaxed, so a ticket might come from what the slot held before
// the word, and the head must not step over a queued step for that.  (An
// acquire before each ticket would do as well: 1024 runs 36.5 -> 37.1 ms, with
// the laps 36.5.)
constexpr int kTicketBits = 18;            // a step's units (kShareUnits) and the late tickets, 8 a CU
CANS_DEV unsigned b2_lap(const Batch2dArgs &b, unsigned idx) { return ((idx >> (31 - __builtin_clz(b.cap))) + 1u) & 63u; }
CANS_DEV void b2_push(const Batch2dArgs &b, int grp, int k, int nunit) {
    Batch2dGroup &g = b.group[grp];
    const unsigned idx = add1(&g.resv, 1u);
    if ((threadIdx.x & 63) == 0)
        __hip_atomic_store(&b.ring[(size_t)grp * b.cap + (idx & (b.cap - 1))],
                           ((unsigned long long)k << 40) | ((unsigned long long)nunit << 24) |
                               ((unsigned long long)b2_lap(b, idx) << kTicketBits),
                           __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    while ((unsigned)uni((int)ald(&g.tail)) != idx) __builtin_amdgcn_s_sleep(1);
    if ((threadIdx.x & 63) == 0)
        (void)__hip_atomic_fetch_add(&g.tail, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}
// What wave 0 found for its workgroup to do: units of its own group's queue,
// else of another's; a step of the workgroup's own run; the next run.
struct B2Do {
    int op, k, unit, grp;
};
CANS_DEV B2Do b2_next(const Batch2dArgs &b, int grp, int NW, bool own) {
    const int lane = threadIdx.x & 63, ng = b.ngroup;
    for (;;) {
        unsigned h = 0, t = 0;
        if (lane < ng) { h = ald(&b.group[lane].head); t = ald(&b.group[lane].tail); }
        const unsigned full = (unsigned)__ballot((int)(t - h) > 0);
        if (full == 0) break;
        const unsigned turned = (full >> grp) | (full << (ng - grp));   // bit 0: the own group
        const int g = (grp + __builtin_ctz(turned)) % ng;
        const unsigned hg = (unsigned)__builtin_amdgcn_readlane((int)h, g);
        const unsigned long long w = add1(&b.ring[(size_t)g * b.cap + (hg & (b.cap - 1))], (unsigned long long)NW);
        const int u = (int)(w & ((1ull << kTicketBits) - 1)), n = (int)((w >> 24) & 0xffffull);
        if (u < n) {
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            return B2Do{B2_UNITS, (int)(w >> 40), u, g};
        }
        const unsigned lap = (unsigned)(w >> kTicketBits) & 63u;
        if (lane == 0 && lap == b2_lap(b, hg)) {   // every unit of the head is taken: the next word
            unsigned want = hg;
            __hip_atomic_compare_exchange_strong(&b.group[g].head, &want, hg + 1u, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (own) return B2Do{B2_OWN, 0, 0, 0};
    unsigned *active = &b.group[0].active;   // shared runs, and workgroups that may be starting one
    if (uni((int)ald(b.next)) < b.nrun) {
        add1(active, 1u);
        // released: who sees the list used up (and acquires) sees this start
        // in `active` too
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        const int q = (int)add1(b.next, 1u);
        if (q < b.nrun) return B2Do{B2_START, b.order ? uni(b.order[q]) : q, 0, q % ng};
        add1(active, ~0u);
    }
    if (uni((int)ald(active)) > 0) return B2Do{B2_IDLE, 0, 0, 0};
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    return B2Do{uni((int)ald(active)) > 0 ? B2_IDLE : B2_EXIT, 0, 0, 0};
}

// The march's arguments of run k for step parity par (0 reads the state and
// writes the scratch, 1 the reverse).
CANS_DEV Mlw2dArgs b2_args(const Batch2dArgs &b, int k, int par) {
    const long long o = uni(b.off[k]), ox = uni(b.offx[k]), oy = uni(b.offy[k]);
    double *in[7], *out[7];
#pragma unroll
    for (int q = 0; q < 7; q++) {
        in[q] = (par ? b.g[q] : b.f[q]) + o;
        out[q] = (par ? b.f[q] : b.g[q]) + o;
    }
    Mlw2dArgs a;
    a.ro = in[0]; a.pr = in[1]; a.vx = in[2]; a.vy = in[3]; a.bx = in[4]; a.by = in[5]; a.az = in[6];
    a.ro_o = out[0]; a.pr_o = out[1]; a.vx_o = out[2]; a.vy_o = out[3]; a.bx_o = out[4]; a.by_o = out[5];
    a.az_o = out[6];
    a.dx = b.dx + ox; a.dxm = b.dxm + ox; a.dy = b.dy + oy; a.dym = b.dym + oy;
    a.mx = Metric{b.mx[0] + ox, b.mx[1] + ox, b.mx[2] + ox, b.mx[3] + ox};
    a.my = Metric{b.my[0] + oy, b.my[1] + oy, b.my[2] + oy, b.my[3] + oy};
    a.qav = b.qav; a.gm = b.gm; a.dt = 0.0; a.clk = nullptr; a.step = 0;
    a.ix = uni(b.ix[k]); a.jx = uni(b.jx[k]);
    a.per_margin = b.margin; a.safety = b.safety; a.peek = 0; a.dt_log = nullptr;
    return a;
}

template <int BT>
__global__ __launch_bounds__(BT) __attribute__((amdgpu_waves_per_eu(kOccBatch))) void batch2d_kernel(Batch2dArgs b) {
    constexpr int NW = BT / 64;
    __shared__ double red[2][NW];
    // the work in hand: a run's step and the units of it, and what came of it
    __shared__ struct { int op, k, grp, u0, u1, nexec, H, nstrip, nunit, end, ns, merr; double dt, t; } c;
    __shared__ struct { int k, ns, nexec, H, nstrip, nunit; double dt, t; } own;   // the workgroup's own run (k >= 0)
    const int wv = uni((int)(threadIdx.x >> 6));
    const int grp = (int)(blockIdx.x % (unsigned)b.ngroup);
    int par = 0;
    if (wv == 0) own.k = -1;
    for (;;) {
        if (wv == 0) {
            const bool have = uni(own.k) >= 0;
            const B2Do d = b2_next(b, grp, NW, have);
            c.op = d.op; c.k = d.k; c.grp = d.grp; c.end = 0;
            if (d.op == B2_UNITS) {
                const Batch2dCtl &r = b.ctl[d.k];
                const int n = uni(ald(&r.nunit));
                c.nexec = uni(ald(&r.nexec)); c.H = uni(ald(&r.H)); c.nstrip = uni(ald(&r.nstrip)); c.nunit = n;
                c.dt = __longlong_as_double(uni((long long)ald(&r.dt_bits)));
                c.u0 = d.unit; c.u1 = min(d.unit + NW, n);
            } else if (d.op == B2_OWN) {
                c.k = own.k; c.nexec = own.nexec; c.H = own.H; c.nstrip = own.nstrip; c.nunit = own.nunit;
                c.dt = own.dt; c.u0 = 0; c.u1 = own.nunit;
            }
        }
        __syncthreads();
        const int op = uni(c.op), k = uni(c.k);
        if (op == B2_EXIT) break;
        if (op == B2_IDLE) {
            __builtin_amdgcn_s_sleep(16);
        } else if (op == B2_START) {
            const long long o = uni(b.off[k]), ox = uni(b.offx[k]), oy = uni(b.offy[k]);
            const int ix = uni(b.ix[k]), jx = uni(b.jx[k]);
            const size_t ncell = (size_t)ix * (size_t)jx;
            // cfl_m of the initial state over every cell (cans2d/common/cfl_m.f:44-62)
            double m = kR4_1e20;
            for (size_t p = threadIdx.x; p < ncell; p += BT) {
                const int i = (int)(p % (size_t)ix) + 1, j = (int)(p / (size_t)ix) + 1;
                const size_t q = (size_t)o + p;
                const double ro = b.f[0][q], pr = b.f[1][q], vx = b.f[2][q], vy = b.f[3][q], bx = b.f[4][q],
                             by = b.f[5][q];
                const double b2 = bx * bx + by * by;
                const double ca2 = b2 * pi4i / ro;
                const double cs2 = b.gm * pr / ro;
                const double v2 = vx * vx + vy * vy;
                const double dtq = b.safety * (fminF(b.dx[ox + i - 1], b.dy[oy + j - 1]) / __builtin_sqrt(v2 + cs2 + ca2));
                if (dtq < m) m = dtq;
            }
            const double dt = block_min<BT>(m, red[par]);
            par ^= 1;
            if (wv == 0) {
                const B2Cut cut = batch2d_cut(ix, jx, NW);
                const bool bad = dt < b.dtmin;                 // cfl_m.f: merr=9001, main.f stops
                const bool share = !bad && cut.nunit > (kShareRounds - 1) * NW && b.nrun < kShareRuns &&
                                   cut.nunit <= kShareUnits;
                if (share) {
                    if (threadIdx.x == 0) {
                        Batch2dCtl &r = b.ctl[k];
                        ast(&r.done, 0u);
                        ast(&r.minkey, (unsigned long long)dkey(kR4_1e20));
                        ast(&r.dt_bits, (unsigned long long)__double_as_longlong(dt));
                        ast(&r.t_bits, (unsigned long long)__double_as_longlong(0.0 + dt));
                        ast(&r.ns, 1); ast(&r.nexec, 0); ast(&r.H, cut.H); ast(&r.nstrip, cut.nstrip);
                        ast(&r.nunit, cut.nunit);
                    }
                    b2_push(b, uni(c.grp), k, cut.nunit);
                } else {
                    add1(&b.group[0].active, ~0u);
                    if (bad) {
                        c.end = 1; c.nexec = 0; c.ns = 1; c.merr = 9001; c.t = 0.0;
                    } else {
                        own.k = k; own.ns = 1; own.nexec = 0; own.dt = dt; own.t = 0.0 + dt;
                        own.H = cut.H; own.nstrip = cut.nstrip; own.nunit = cut.nunit;
                    }
                }
            }
        } else {   // a step of the own run, or units of a shared run's step
            {
                const int nstrip = uni(c.nstrip), u1 = uni(c.u1), H = uni(c.H);
                const double dt = uni(c.dt);
                const Mlw2dArgs a = b2_args(b, k, uni(c.nexec) & 1);
                const YMet<KPtr> y{(KPtr)a.my.dim, (KPtr)a.my.di, (KPtr)a.my.u0, (KPtr)a.my.u1, (KPtr)a.dym, (KPtr)a.dy};
                double dmin = kR4_1e20;
                for (int u = uni(c.u0) + wv; u < u1; u += NW)
                    march_strip(a, PerBox{}, y, H, u % nstrip, u / nstrip, dt, true, dmin);
                red[par][wv] = wave_min(dmin);
            }
            __builtin_amdgcn_s_waitcnt(0x0f70);   // this wave's stores have reached L2 (vmcnt 0)
            __syncthreads();                      // (the own run's step ends here)
            if (wv == 0) {
                const double m = read_lane(row_min15(red[par][threadIdx.x & (NW - 1)]), 15);
                Batch2dCtl &r = b.ctl[k];
                const bool mine = op == B2_OWN;
                const int u0 = uni(c.u0), u1 = uni(c.u1), nunit = uni(c.nunit), nexec = uni(c.nexec) + 1;
                const unsigned cnt = (unsigned)(u1 - u0);
                unsigned d = 0;
                if (!mine && threadIdx.x == 0) {
                    atomicMin(&r.minkey, (unsigned long long)dkey(m));
                    d = __hip_atomic_fetch_add(&r.done, cnt, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
                }
                if ((unsigned)uni((int)d) + cnt == (unsigned)nunit) {   // the step's last units: its end and the next
                    const double dt = mine ? m : dunkey((unsigned long long)uni((long long)ald(&r.minkey)));
                    double t = mine ? own.t : __longlong_as_double(uni((long long)ald(&r.t_bits)));
                    int ns = uni(mine ? own.ns : ald(&r.ns));
                    const bool more = ns < b.nstop && uni(t) < b.tend;
                    if (more) ns++;
                    const bool bad = more && uni(dt) < b.dtmin;
                    if (more && !bad) {
                        t = t + dt;
                        if (mine) {
                            own.ns = ns; own.nexec = nexec; own.dt = dt; own.t = t;
                        } else {
                            if (threadIdx.x == 0) {
                                ast(&r.done, 0u);
                                ast(&r.minkey, (unsigned long long)dkey(kR4_1e20));
                                ast(&r.dt_bits, (unsigned long long)__double_as_longlong(dt));
                                ast(&r.t_bits, (unsigned long long)__double_as_longlong(t));
                                ast(&r.ns, ns); ast(&r.nexec, nexec);
                            }
                            b2_push(b, uni(c.grp), k, nunit);
                        }
                    } else {
                        c.end = 1; c.nexec = nexec; c.ns = ns; c.merr = bad ? 9001 : 0; c.t = t;
                        if (mine) own.k = -1;
                        else add1(&b.group[0].active, ~0u);
                    }
                }
            }
            par ^= 1;
        }
        __syncthreads();
        if (uni(c.end)) {
            if (uni(c.nexec) & 1) {   // the last state is in the scratch set: copy back
                const long long o = uni(b.off[k]);
                const size_t ncell = (size_t)uni(b.ix[k]) * (size_t)uni(b.jx[k]);
                for (size_t p = threadIdx.x; p < ncell; p += BT)
#pragma unroll
                    for (int q = 0; q < 7; q++) b.f[q][(size_t)o + p] = b.g[q][(size_t)o + p];
            }
            if (wv == 0) {   // uniform branch; the lanes store identical values
                b.t_out[k] = c.t;
                b.ns_out[k] = c.ns;
                b.merr_out[k] = c.merr;
            }
            __syncthreads();   // every wave has read c before wave 0 writes it again
        }
    }
}

// per-run metric of both axes (the arithmetic of the single-run metric
// kernel) by block r for run r; the queue counters, and the rings empty
__global__ void batch2d_prep(Batch2dArgs b) {
    const int r = blockIdx.x;
    const size_t nw = (size_t)b.ngroup * b.cap, step = (size_t)gridDim.x * blockDim.x;
    for (size_t p = (size_t)r * blockDim.x + threadIdx.x; p < nw; p += step) b.ring[p] = 0ull;
    if (r == 0) {
        if (threadIdx.x == 0) *b.next = 0u;
        if ((int)threadIdx.x < b.ngroup) {
            Batch2dGroup &g = b.group[threadIdx.x];
            g.head = g.tail = g.resv = g.active = 0u;
        }
    }
    if (r >= b.nrun) return;
    for (int axis = 0; axis < 2; axis++) {
        const long long o = axis ? b.offy[r] : b.offx[r];
        const int n = axis ? b.jx[r] : b.ix[r];
        const double *d = (axis ? b.dy : b.dx) + o, *dm = (axis ? b.dym : b.dxm) + o;
        double *const *m = axis ? b.my : b.mx;
        for (int i = 1 + (int)threadIdx.x; i <= n; i += blockDim.x) {
            m[0][o + i - 1] = 1.0 / d[i - 1];
            m[1][o + i - 1] = 1.0 / dm[i - 1];
            if (i >= 2 && i <= n - 1) {
                m[2][o + i - 1] = 0.5 * dm[i - 1] / d[i - 1];
                m[3][o + i - 1] = 0.5 * dm[i - 2] / d[i - 1];
            } else {
                m[2][o + i - 1] = 0.0;
                m[3][o + i - 1] = 0.0;
            }
        }
    }
}

constexpr int kOcc = 2;   // waves per SIMD the register budget is compiled for

}  // namespace

hipError_t launch_batch2d(const Batch2dArgs &b, int block_threads, int nblocks, hipStream_t s) {
    hipLaunchKernelGGL(batch2d_prep, dim3(b.nrun > 64 ? b.nrun : 64), dim3(256), 0, s, b);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || b.nrun == 0) return e;
    switch (block_threads) {
    case 64: hipLaunchKernelGGL(batch2d_kernel<64>, dim3(nblocks), dim3(64), 0, s, b); break;
    case 128: hipLaunchKernelGGL(batch2d_kernel<128>, dim3(nblocks), dim3(128), 0, s, b); break;
    case 256: hipLaunchKernelGGL(batch2d_kernel<256>, dim3(nblocks), dim3(256), 0, s, b); break;
    case 512: hipLaunchKernelGGL(batch2d_kernel<512>, dim3(nblocks), dim3(512), 0, s, b); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_mlw2d(const Mlw2dArgs &a, hipStream_t s, const BndMap *map) {
    if (a.ix < 3 || a.jx < 3) return hipSuccess;
    const int h = pick_rows(a.ix, a.jx);
    const int nstrip = (a.ix - 2 + COLS - 1) / COLS;
    const int nrowb = (a.jx - 2 + h - 1) / h;
    const int nblocks = (nstrip * nrowb + WPB - 1) / WPB;
    if (map) {
        const Faces f = pack_faces(*map);
        hipLaunchKernelGGL((mlw2d_kernel<kOcc, Faces>), dim3(nblocks), dim3(WAVE * WPB), 0, s, a, f, h, a.my.dim,
                           a.my.di, a.my.u0, a.my.u1, a.dym, a.dy);
    } else {
        hipLaunchKernelGGL((mlw2d_kernel<kOcc, PerBox>), dim3(nblocks), dim3(WAVE * WPB), 0, s, a, PerBox{}, h,
                           a.my.dim, a.my.di, a.my.u0, a.my.u1, a.dym, a.dy);
    }
    return hipGetLastError();
}

}  // namespace cans

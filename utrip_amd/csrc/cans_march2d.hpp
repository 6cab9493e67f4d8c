// cans_march2d.hpp -- what the 2D marching kernels share (cans_mlw2d.hip,
// cans_mlw2d_m3.hip): a wave owns a strip of 64 columns, one of them a halo
// on each side, and marches along y with the stencil rows in registers and
// the x neighbours in the adjacent lanes.
#pragma once
#include "cans_common.hpp"
#include "cans_kernels.hpp"
#include "cans_wave.hpp"

namespace cans {
namespace march2d {

constexpr int WAVE = 64;
constexpr int COLS = WAVE - 2;               // output columns per wave
constexpr int WPB = 4;                       // waves per block
constexpr double pi8i = 1.0 / kPi / 8.0;     // mlw_m.f:27  pi8i=1./pi/8.
constexpr double pi4i = 1.0 / kPi / 4.0;     // mlw_m.f:28  pi4i=1./pi/4.

// x neighbours: shl1/shr1 of cans_wave.hpp (lane l receives lane l+1 / l-1
// through a DPP wave shift; the edge lanes receive 0, and their results are
// never used by an output lane).

// Where the ghost images of a cell lie: PerBox, the periodic box of the
// plain resident run (the benchmark's; its code has no look-ups), or Faces, a
// BndMap packed into three words: per face (axis * 2 + side) two bits of
// kinds, and sixteen of its axis' neg.
struct PerBox {};
struct Faces {
    unsigned kinds, neg[2];
    CANS_DEV int kind(int axis, int side) const { return (int)(kinds >> (4 * axis + 2 * side)) & 3; }
    CANS_DEV unsigned sign(int axis, int side) const { return (neg[axis] >> (16 * side)) & 0xffffu; }
    // the same words, opaque to the compiler: the rare rows and strips at an
    // edge unpack them there instead of holding the pieces through the march
    CANS_DEV Faces here() const {
        Faces f = *this;
        asm volatile("" : "+s"(f.kinds), "+s"(f.neg[0]), "+s"(f.neg[1]));
        return f;
    }
};
template <class M> inline constexpr bool kMapped = false;
template <> inline constexpr bool kMapped<Faces> = true;

// The ghost cells of one axis (n cells, width m) that are copies of cell i:
// lo_n from lo_t up on the low side, hi_n from hi_t up on the high side.
struct Images {
    int lo_n, lo_t, hi_n, hi_t;
    CANS_DEV int count() const { return lo_n + hi_n; }
    CANS_DEV int at(int k) const { return k < lo_n ? lo_t + k : hi_t + k - lo_n; }
};
CANS_DEV Images images_of(const Faces &b, int axis, int i, int n, int m) {
    Images r{0, 0, 0, 0};
    const int lo = b.kind(axis, 0), hi = b.kind(axis, 1), e = n - m;
    if (lo == BM_FRE) { r.lo_t = 1; r.lo_n = i == m + 1 ? m : 0; }                                     // bdfrex.f
    else if (lo == BM_SP) { r.lo_t = 2 * m + 1 - i; r.lo_n = i >= m + 1 && i <= 2 * m; }               // bdsppx.f
    else if (lo == BM_SM) { r.lo_t = 2 * m + 2 - i; r.lo_n = i >= m + 2 && i <= 2 * m + 1; }           // bdsmpx.f
    else { r.lo_t = i - (n - 2 * m); r.lo_n = i >= n - 2 * m + 1 && i <= e; }                          // bdperx.f
    if (hi == BM_FRE) { r.hi_t = e + 1; r.hi_n = i == e ? m : 0; }
    else if (hi == BM_SP) { r.hi_t = 2 * e + 1 - i; r.hi_n = i >= e - m + 1 && i <= e; }
    else if (hi == BM_SM) { r.hi_t = 2 * e - i; r.hi_n = i >= e - m && i <= e - 1; }
    else { r.hi_t = i + (n - 2 * m); r.hi_n = i >= m + 1 && i <= 2 * m; }
    return r;
}
// smallest of d at cell i and at its images
template <class P>
CANS_DEV double images_min(const Faces &b, int axis, P d, int i, int n, int m) {
    double g = d[i - 1];
    const Images r = images_of(b, axis, i, n, m);
    for (int k = 0; k < r.count(); k++) g = fminF(g, d[r.at(k) - 1]);
    return g;
}

// Per-row (y) constants: non-aliased kernel arguments (const double *) in the
// single-run kernel, constant address space in the batched one, so that the
// uniform loads are scalar.
template <class P> struct YMet {
    P dim, di, u0, u1, dym, dy;
};
typedef const __attribute__((address_space(4))) double *KPtr;

// Per-column constants of a strip.
struct ColCtx {
    int i;
    bool out;                     // output column
    unsigned boff;                // byte offset of column min(i,ix) within a row
    double dxi, dxim, dxim1;      // 1/dx(i), 1/dxm(i), 1/dxm(i-1)
    double ux0, ux1;              // 0.5*dxm(i)/dx(i), 0.5*dxm(i-1)/dx(i)
    double qxs;                   // qav*dxm(i)
    double dxc;                   // dx(i)
    double dxg;                   // min of dx(i) and dx of i's x images
    bool edge;                    // mapped: a column of the strip has x images (uniform)
};

// Row j (clamped to the grid, so every lane reads a real cell) of a field:
// a wave-uniform base address plus the lane's 32-bit byte offset.
CANS_DEV const double *row_of(const double *f, int ix, int jx, int j) {
    const int jc = j < 1 ? 1 : (j > jx ? jx : j);
    return f + (size_t)(jc - 1) * (size_t)ix;
}
CANS_DEV double ld(const double *row, unsigned boff) {
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(row) + boff);
}
CANS_DEV void st(double *row, unsigned boff, double v) {
    *reinterpret_cast<double *>(reinterpret_cast<char *>(row) + boff) = v;
}

// one conserved component of the corner half step (mlwhalf.f:47-50):
// A=(i,j) B=(i+1,j) C=(i,j+1) D=(i+1,j+1)
CANS_DEV double half1(double uA, double uB, double uC, double uD, double fA, double fB, double fC, double fD,
                      double gA, double gB, double gC, double gD, double dxim, double dyim, double dt) {
    const double uh = 0.25 * (uB + uA + uD + uC);
    const double dfdx = dxim * (fB - fA + fD - fC) / 2.0;
    const double dfdy = dyim * (gC - gA + gD - gB) / 2.0;
    return uh - dt * dfdx - dt * dfdy;
}

// bx has no x flux and by no y flux.  The reference still forms the zero
// term, dt*(dm*(+0)/2) = +0 for finite dt >= 0 and positive metric, and
// subtracting +0 leaves every value (-0 included) unchanged: these variants
// omit it and give the same bits.
CANS_DEV double half1_y(double uA, double uB, double uC, double uD, double gA, double gB, double gC, double gD,
                        double dyim, double dt) {
    const double uh = 0.25 * (uB + uA + uD + uC);
    const double dfdy = dyim * (gC - gA + gD - gB) / 2.0;
    return uh - dt * dfdy;
}
CANS_DEV double half1_x(double uA, double uB, double uC, double uD, double fA, double fB, double fC, double fD,
                        double dxim, double dt) {
    const double uh = 0.25 * (uB + uA + uD + uC);
    const double dfdx = dxim * (fB - fA + fD - fC) / 2.0;
    return uh - dt * dfdx;
}

CANS_DEV double av_coef(double qs, double vhi, double vlo) {   // mlw_m.f:276-288
    const double zero = 0.0;
    return qs * fmaxF(zero, __builtin_fabs(vhi - vlo) - kR4_1em4);
}

// du of one equation: centre term of mlwhalf (mlwhalf.f:36-41), mlwfull
// (mlwfull.f:31-41) and mlwartv (mlwartv.f:33-41), in the reference's order.
//   dfx = fE-fW   dgy = gN-gS   hS/hN = corner x differences south/north
//   kW/kE = corner y differences west/east   dE = uE-uc  dW = uc-uW
//   dN = uN-uc   dS = uc-uS
struct RowCoef {
    double hdt, dt;               // 0.5*dt, dt
    double hdxi, dxi, hdyi, dyi;  // 0.5/dx(i), 1/dx(i), 0.5/dy(j), 1/dy(j)
    double ux0, ux1, uy0, uy1;
    double qxe, qxw, qyn, qys;    // qxc*dxim, qxw*dxim1, qyc*dyim, qys*dyim1
};

CANS_DEV double du1(const RowCoef &r, double dfx, double dgy, double hS, double hN, double kW, double kE, double dE,
                    double dW, double dN, double dS) {
    double du = 0.0;
    du = du - r.hdt * (r.hdxi * dfx) - r.hdt * (r.hdyi * dgy);
    const double dfdx = r.dxi * (r.uy0 * hS + r.uy1 * hN);
    const double dfdy = r.dyi * (r.ux0 * kW + r.ux1 * kE);
    du = du - r.hdt * dfdx - r.hdt * dfdy;
    du = du + r.dt * (r.dxi * (r.qxe * dE - r.qxw * dW)) + r.dt * (r.dyi * (r.qyn * dN - r.qys * dS));
    return du;
}

// bx (no x flux) and by (no y flux): the zero-flux terms of du1 are +0 for
// finite dt >= 0 and positive metric and are omitted (same bits).
CANS_DEV double du1_y(const RowCoef &r, double dgy, double kW, double kE, double dE, double dW, double dN,
                      double dS) {
    double du = 0.0;
    du = du - r.hdt * (r.hdyi * dgy);
    const double dfdy = r.dyi * (r.ux0 * kW + r.ux1 * kE);
    du = du - r.hdt * dfdy;
    du = du + r.dt * (r.dxi * (r.qxe * dE - r.qxw * dW)) + r.dt * (r.dyi * (r.qyn * dN - r.qys * dS));
    return du;
}
CANS_DEV double du1_x(const RowCoef &r, double dfx, double hS, double hN, double dE, double dW, double dN,
                      double dS) {
    double du = 0.0;
    du = du - r.hdt * (r.hdxi * dfx);
    const double dfdx = r.dxi * (r.uy0 * hS + r.uy1 * hN);
    du = du - r.hdt * dfdx;
    du = du + r.dt * (r.dxi * (r.qxe * dE - r.qxw * dW)) + r.dt * (r.dyi * (r.qyn * dN - r.qys * dS));
    return du;
}

// The strip's column of this lane and its constants.
template <class A, class M>
CANS_DEV ColCtx column_of(const A &a, const M &map, int strip) {
    const int ix = a.ix, lane = threadIdx.x & (WAVE - 1);
    ColCtx x;
    x.i = 1 + strip * COLS + lane;         // lane 0 is the west halo column
    x.out = lane >= 1 && lane <= COLS && x.i <= ix - 1 &&
            (a.per_margin == 0 || (x.i >= a.per_margin + 1 && x.i <= ix - a.per_margin));
    const int ic = min(x.i, ix);           // lanes past the grid read column ix
    x.boff = (unsigned)(ic - 1) * 8u;
    x.dxi = a.mx.di[ic - 1];
    x.dxim = a.mx.dim[ic - 1];
    x.dxim1 = a.mx.dim[max(ic - 2, 0)];
    x.ux0 = a.mx.u0[ic - 1];
    x.ux1 = a.mx.u1[ic - 1];
    x.qxs = a.qav * a.dxm[ic - 1];
    x.dxc = a.dx[ic - 1];
    x.dxg = x.dxc;
    if constexpr (kMapped<M>) {
        const int mg = a.per_margin;
        x.edge = strip * COLS < 2 * mg + 1 || (strip + 1) * COLS + 1 >= ix - 2 * mg;
        x.dxg = images_min(map, 0, a.dx, ic, ix, mg);
    } else {
        const int mg = a.per_margin;
        if (mg > 0 && ic >= ix - 2 * mg + 1) x.dxg = fminF(x.dxg, a.dx[ic - (ix - 2 * mg) - 1]);
        if (mg > 0 && ic <= 2 * mg) x.dxg = fminF(x.dxg, a.dx[ic + (ix - 2 * mg) - 1]);
    }
    return x;
}

constexpr int kWaveSlots = 256 * 4 * 2;    // two waves on each SIMD of the 256 CUs
// Rows per wave.  Each wave pays about 1.5 rows of prologue, and a row takes
// about 2.0 us for a wave that has its SIMD to itself and 3.3 us for each of
// two that share one (FP64 latency against FP64 issue), so the launch's cost
// is (H + 1.5) * (3.3 per full round of 2048 waves, plus 2.0 or 3.3 for the
// rest by whether it has more waves than SIMDs).  Small grids so take short
// strips, many waves deep across the chip: whole steps with 8 rows at least
// and with this rule, 64^2 22.8 -> 9.0 us (1 row), 256^2 23.2 -> 13.1 (2),
// 512^2 23.2 -> 17.1 (5), 700^2 30.9 -> 25.9 (9), 2000x300 31.3 -> 25.7 (5);
// 1024^2 (9 rows) and up as before.
inline int pick_rows(int ix, int jx) {
    const long nstrip = (ix - 2 + COLS - 1) / COLS;
    constexpr double kAlone = 2.0, kShared = 3.3;   // us per row
    int best = 16;
    double cost = 1e300;
    for (int h = 1; h <= 96; h++) {
        const long waves = nstrip * ((jx - 2 + h - 1) / h);
        const long full = waves / kWaveSlots, rest = waves % kWaveSlots;
        const double c = (h + 1.5) * (full * kShared + (rest == 0 ? 0.0 : (rest <= kWaveSlots / 2 ? kAlone : kShared)));
        if (c < cost) { cost = c; best = h; }
    }
    return best;
}

inline Faces pack_faces(const BndMap &map) {
    Faces f{0, {0, 0}};
    for (int d = 0; d < 2; d++)
        for (int side = 0; side < 2; side++) {
            f.kinds |= (unsigned)map.kind[d][side] << (4 * d + 2 * side);
            f.neg[d] |= map.neg[d][side] << (16 * side);
        }
    return f;
}

}  // namespace march2d
}  // namespace cans

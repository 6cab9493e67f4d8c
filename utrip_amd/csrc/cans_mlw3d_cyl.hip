// cans_mlw3d_cyl.hip -- the 3D modified Lax-Wendroff step on a cylindrical
// grid (r, phi, z), cans3d/hdmlw/mlw_m_c.f:2-520 with mlwhalf.f:38-68,
// mlwsrch.f:33-46, mlwfull.f:34-55, mlwsrcf.f:33-46 and mlwartv.f:36-48, on
// gfx950, bit-exact FP64.
//
// Two kernels, the corner values between them in HBM (26 a corner: fluxes,
// the phi ones divided by the radius, and the geometric sources):
//   corners  a block of 64 x 8 threads (on grids narrow in x 16 x 32 or 8 x 64)
//            marches an (x, y) tile of cells in z.
//            Each step turns the primitives of a plane into the 39 cell
//            values (LDS), and forms the 63 x 7 corners below it from the
//            cells of the plane and from what its own thread kept of the
//            plane before: sums that run over the lower plane's four cells
//            and then the upper one's are continued where they stopped.
//            Only the z fluxes, which alternate between the planes, are kept
//            in LDS for two planes.  159,744 bytes a block, 2 waves a SIMD.
//   update   a thread per cell.  The cell values it needs of itself and its
//            six neighbours it forms again from the primitives, 56 loads
//            against 104 of stored cell values.
// 160 x 64 x 128 cells, a step with cfl and fill: 644 -> 382 us against three
// kernels that also passed 32 values a cell through HBM (95 + 233 + 248 us).
#include "cans_clock.hpp"
#include "cans_common.hpp"
#include "cans_roe.hpp"

namespace cans {
namespace {

constexpr double pi8i = 1.0 / kPi / 8.0;
constexpr double pi4i = 1.0 / kPi / 4.0;
constexpr int CNT = 512;   // cells of a tile plane, CTX x CNT / CTX of them; threads of a block

// corner scratch slots (mlw_m_c.f:273-408): x fluxes, E, phi fluxes / xm, z
// fluxes, sources
enum { Z_ROX, Z_EEX, Z_RXX, Z_RYX, Z_RZX, Z_EX, Z_EY, Z_EZ,
       Z_FRO, Z_FEE, Z_FRX, Z_FRY, Z_FRZ, Z_FBX, Z_FBZ,
       Z_ROZ, Z_EEZ, Z_RXZ, Z_RYZ, Z_RZZ,
       Z_SRO, Z_SEE, Z_SRX, Z_SRY, Z_SRZ, Z_SBZ, Z_NCORN };
static_assert(Z_NCORN == kMlw3dCylCornerFields, "cylindrical corner slots");

// One state's values: u = ro ee rx ry rz bx by bz; fluxes x, phi (divided by
// the radius r) and z; sources of ro ee rx ry rz bz (mlw_m_c.f:109-243 at
// cells, :273-408 at corners).  Unused members cost nothing.
struct Vals {
    double eex, rxx, ryx, rzx, ex, ey, ez;
    double fro, fee, frx, fry, frz, fbx, fbz;
    double roz, eez, rxz, ryz, rzz;
    double rox;
    double src[6];
};
struct State {
    double ro, pr, vx, vy, vz, bx, by, bz;
};
CANS_DEV void conserved(const State &w, double gm, double *u) {
    const double vv = w.vx * w.vx + w.vy * w.vy + w.vz * w.vz;
    const double bb = w.bx * w.bx + w.by * w.by + w.bz * w.bz;
    u[0] = w.ro;
    u[1] = w.pr / (gm - 1.0) + 0.5 * w.ro * vv + pi8i * bb;
    u[2] = w.ro * w.vx;
    u[3] = w.ro * w.vy;
    u[4] = w.ro * w.vz;
    u[5] = w.bx;
    u[6] = w.by;
    u[7] = w.bz;
}
CANS_DEV double vals_ep(const State &w, double gm) {
    const double vv = w.vx * w.vx + w.vy * w.vy + w.vz * w.vz;
    return w.pr * gm / (gm - 1.0) + 0.5 * w.ro * vv;
}
CANS_DEV void vals_e(const State &w, Vals &f) {
    f.ex = -w.vy * w.bz + w.vz * w.by;
    f.ey = -w.vz * w.bx + w.vx * w.bz;
    f.ez = -w.vx * w.by + w.vy * w.bx;
}
CANS_DEV void vals_x(const State &w, double gm, Vals &f) {
    vals_e(w, f);
    f.rox = w.ro * w.vx;
    f.eex = vals_ep(w, gm) * w.vx + (w.bz * f.ey - w.by * f.ez) * pi4i;
    f.rxx = w.ro * (w.vx * w.vx) + w.pr + pi8i * (w.by * w.by + w.bz * w.bz - w.bx * w.bx);
    f.ryx = w.ro * w.vy * w.vx - pi4i * w.by * w.bx;
    f.rzx = w.ro * w.vz * w.vx - pi4i * w.bz * w.bx;
}
CANS_DEV void vals_y(const State &w, double gm, double r, Vals &f) {
    vals_e(w, f);
    f.fro = w.ro * w.vy / r;
    f.fee = (vals_ep(w, gm) * w.vy + (w.bx * f.ez - w.bz * f.ex) * pi4i) / r;
    f.frx = (w.ro * w.vx * w.vy - pi4i * w.bx * w.by) / r;
    f.fry = (w.ro * (w.vy * w.vy) + w.pr + pi8i * (w.bx * w.bx + w.bz * w.bz - w.by * w.by)) / r;
    f.frz = (w.ro * w.vz * w.vy - pi4i * w.bz * w.by) / r;
    f.fbx = f.ez / r;
    f.fbz = -f.ex / r;
}
CANS_DEV void vals_z(const State &w, double gm, Vals &f) {
    vals_e(w, f);
    f.roz = w.ro * w.vz;
    f.eez = vals_ep(w, gm) * w.vz + (w.by * f.ex - w.bx * f.ey) * pi4i;
    f.rxz = w.ro * w.vx * w.vz - pi4i * w.bx * w.bz;
    f.ryz = w.ro * w.vy * w.vz - pi4i * w.by * w.bz;
    f.rzz = w.ro * (w.vz * w.vz) + w.pr + pi8i * (w.bx * w.bx + w.by * w.by - w.bz * w.bz);
}
// needs the x fluxes and E; p4r = pi4i / r, p8r = 2 * pi4i / r
CANS_DEV void vals_src(const State &w, double r, double p4r, double p8r, Vals &f) {
    f.src[0] = -(f.rox / r);
    f.src[1] = -(f.eex / r);
    f.src[2] = -(w.ro / r * (w.vx * w.vx - w.vy * w.vy)) + p4r * (w.bx * w.bx - w.by * w.by);
    f.src[3] = -(2.0 * w.ro / r * w.vx * w.vy) + p8r * w.bx * w.by;
    f.src[4] = -(f.rzx / r);
    f.src[5] = -(f.ey / r);
}

// flux of equation q by direction; bx has no x flux, by no phi flux, bz no z
// flux (constant q: resolved at compile time)
CANS_DEV double xflux(const Vals &f, int q) {
    switch (q) {
    case 0: return f.rox;
    case 1: return f.eex;
    case 2: return f.rxx;
    case 3: return f.ryx;
    case 4: return f.rzx;
    case 6: return -f.ez;
    case 7: return f.ey;
    default: return 0.0;
    }
}
CANS_DEV double yflux(const Vals &f, int q) {
    switch (q) {
    case 0: return f.fro;
    case 1: return f.fee;
    case 2: return f.frx;
    case 3: return f.fry;
    case 4: return f.frz;
    case 5: return f.fbx;
    case 7: return f.fbz;
    default: return 0.0;
    }
}
CANS_DEV double zflux(const Vals &f, int q) {
    switch (q) {
    case 0: return f.roz;
    case 1: return f.eez;
    case 2: return f.rxz;
    case 3: return f.ryz;
    case 4: return f.rzz;
    case 5: return -f.ey;
    case 6: return f.ex;
    default: return 0.0;
    }
}
__device__ constexpr int kSrc[8] = {0, 1, 2, 3, 4, -1, -1, 5};   // source of each equation

// LDS slots of a cell plane; the z part for two planes
enum { L_RO, L_EE, L_RX, L_RY, L_BX, L_BY, L_BZ, L_EEX, L_RXX, L_RYX, L_RZX, L_EZ, L_FY, L_SRC = L_FY + 7,
       L_N = L_SRC + 6 };
enum { M_RZ, M_EEZ, M_RXZ, M_RYZ, M_RZZ, M_EY, M_EX, M_N };
struct Plane {
    double c[L_N][CNT];
    double z[2][M_N][CNT];
};
static_assert(sizeof(Plane) == 159744, "one block a CU");

CANS_DEV double pu(const Plane &L, int par, int q, int t) {
    switch (q) {
    case 4: return L.z[par][M_RZ][t];
    case 5: return L.c[L_BX][t];
    case 6: return L.c[L_BY][t];
    case 7: return L.c[L_BZ][t];
    default: return L.c[L_RO + q][t];
    }
}
CANS_DEV double px(const Plane &L, int par, int q, int t) {
    switch (q) {
    case 0: return L.c[L_RX][t];
    case 1: return L.c[L_EEX][t];
    case 2: return L.c[L_RXX][t];
    case 3: return L.c[L_RYX][t];
    case 4: return L.c[L_RZX][t];
    case 6: return -L.c[L_EZ][t];
    case 7: return L.z[par][M_EY][t];
    default: return 0.0;
    }
}
CANS_DEV double py(const Plane &L, int q, int t) { return q == 6 ? 0.0 : L.c[L_FY + (q == 7 ? 6 : q)][t]; }
CANS_DEV double pz(const Plane &L, int par, int q, int t) {
    switch (q) {
    case 5: return -L.z[par][M_EY][t];
    case 6: return L.z[par][M_EX][t];
    case 7: return 0.0;
    default: return L.z[par][M_RZ + q][t];
    }
}

CANS_DEV double ld(const double *plane, unsigned boff) {
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(plane) + boff);
}
CANS_DEV void st(double *plane, unsigned boff, double v) {
    *reinterpret_cast<double *>(reinterpret_cast<char *>(plane) + boff) = v;
}

CANS_DEV bool cyl_dt(const Mlw3dArgs &a, double &dt) {   // after the step's clock kernel
    if (!a.clk) { dt = a.dt; return true; }
    const StepCtl c = clock_peek(a.clk, a.step);
    dt = c.dt;
    return c.run;
}

// Corners [k0, k1) of the tile (corner k between the cell planes k and k+1,
// 0-based), wx x wy of them a plane: the tiles of a row or column have equal
// widths, since a last one of a few columns, whose rows are stores of less
// than 64 bytes, took twice as long as the others (64 columns of 30 x 157
// corners: 111 -> 50 us; the cell and corner kernels before 52).
template <int CTX>
__global__ __launch_bounds__(CNT) __attribute__((amdgpu_waves_per_eu(2, 2))) void cyl_corners(Mlw3dArgs a, int wx, int wy,
                                                                                             int tiles_x, int ntiles,
                                                                                             int nseg, int seglen) {
    constexpr int CTY = CNT / CTX;
    static_assert(CNT % CTX == 0 && CTY > 1, "tile shape");
    const unsigned per = gridDim.x / kXcds;
    const int item = (int)((blockIdx.x % kXcds) * per + blockIdx.x / kXcds);
    if (item >= ntiles * nseg) return;
    double dt;
    if (!cyl_dt(a, dt)) return;   // uniform across the launch
    __shared__ Plane L;
    const int ix = a.ix, jx = a.jx, kx = a.kx;
    const int tile = item % ntiles;
    const int k0 = (item / ntiles) * seglen;
    const int k1 = min(kx - 1, k0 + seglen);
    const double gm = a.gm;
    const int t = threadIdx.x, ti = t % CTX, tj = t / CTX;
    const int gx = (tile % tiles_x) * wx + ti;   // 0-based cell of this thread
    const int gy = (tile / tiles_x) * wy + tj;
    const bool cval = ti <= wx && tj <= wy && gx < ix && gy < jx;
    const bool kval = ti < wx && tj < wy && gx <= ix - 2 && gy <= jx - 2;
    const size_t N = (size_t)ix * jx * kx, sz = (size_t)ix * jx;
    const size_t p0 = cval ? (size_t)gx + (size_t)ix * gy : 0;
    const double r = cval ? a.x[gx] : 1.0, rm = kval ? a.xm[gx] : 1.0;
    const double p4r = pi4i / r, p8r = 2.0 * pi4i / r, p4rm = pi4i / rm, p8rm = 2.0 * pi4i / rm;
    const double dxim = kval ? a.mx.dim[gx] : 0.0, dyim = kval ? a.my.dim[gy] : 0.0;
    double uhp[8], fxp[8], fyp[8], shp[6];   // lower plane's part of the corner's sums
#pragma unroll
    for (int q = 0; q < 8; q++) uhp[q] = fxp[q] = fyp[q] = 0.0;
#pragma unroll
    for (int q = 0; q < 6; q++) shp[q] = 0.0;
    // scalar plane base + 32-bit lane offset; opaque in the loop, where the
    // compiler would otherwise hold 34 64-bit field addresses a lane
    unsigned boff = (unsigned)p0 * 8u;
    double nxt[8];
    if (cval) {
#pragma unroll
        for (int f = 0; f < 8; f++) nxt[f] = ld(a.prim[f] + sz * k0, boff);
    }
    // the cell values of plane s, its primitives loaded; those of plane s+1 under way
    auto put_plane = [&](int s) {
        const int par = s & 1;
        asm volatile("" : "+v"(boff));
        if (!cval) return;
        const State w{nxt[0], nxt[1], nxt[2], nxt[3], nxt[4], nxt[5], nxt[6], nxt[7]};
        if (s < k1) {
#pragma unroll
            for (int f = 0; f < 8; f++) nxt[f] = ld(a.prim[f] + sz * (s + 1), boff);
        }
        double u[8];
        Vals f;
        conserved(w, gm, u);
        vals_x(w, gm, f);
        vals_y(w, gm, r, f);
        vals_z(w, gm, f);
        vals_src(w, r, p4r, p8r, f);
        L.c[L_RO][t] = u[0];
        L.c[L_EE][t] = u[1];
        L.c[L_RX][t] = u[2];
        L.c[L_RY][t] = u[3];
        L.c[L_BX][t] = u[5];
        L.c[L_BY][t] = u[6];
        L.c[L_BZ][t] = u[7];
        L.c[L_EEX][t] = f.eex;
        L.c[L_RXX][t] = f.rxx;
        L.c[L_RYX][t] = f.ryx;
        L.c[L_RZX][t] = f.rzx;
        L.c[L_EZ][t] = f.ez;
        L.c[L_FY + 0][t] = f.fro;
        L.c[L_FY + 1][t] = f.fee;
        L.c[L_FY + 2][t] = f.frx;
        L.c[L_FY + 3][t] = f.fry;
        L.c[L_FY + 4][t] = f.frz;
        L.c[L_FY + 5][t] = f.fbx;
        L.c[L_FY + 6][t] = f.fbz;
#pragma unroll
        for (int q = 0; q < 6; q++) L.c[L_SRC + q][t] = f.src[q];
        L.z[par][M_RZ][t] = u[4];
        L.z[par][M_EEZ][t] = f.eez;
        L.z[par][M_RXZ][t] = f.rxz;
        L.z[par][M_RYZ][t] = f.ryz;
        L.z[par][M_RZZ][t] = f.rzz;
        L.z[par][M_EY][t] = f.ey;
        L.z[par][M_EX][t] = f.ex;
    };
    // the first plane is only a lower one
    put_plane(k0);
    __syncthreads();
    if (kval) {
        const int par = k0 & 1, t1 = t + 1, t2 = t + CTX, t3 = t + CTX + 1;   // cells 10, 01, 11 of the corner
#pragma unroll
        for (int q = 0; q < 8; q++) {
            uhp[q] = pu(L, par, q, t1) + pu(L, par, q, t) + pu(L, par, q, t3) + pu(L, par, q, t2);
            if (q != 5) fxp[q] = px(L, par, q, t1) - px(L, par, q, t) + px(L, par, q, t3) - px(L, par, q, t2);
            if (q != 6) fyp[q] = py(L, q, t2) - py(L, q, t) + py(L, q, t3) - py(L, q, t1);
        }
#pragma unroll
        for (int e = 0; e < 6; e++) {
            const double *c = L.c[L_SRC + e];
            shp[e] = c[t1] + c[t] + c[t3] + c[t2];
        }
    }
    __syncthreads();
    for (int s = k0 + 1; s <= k1; s++) {
        const int par = s & 1, lp = par ^ 1;
        put_plane(s);
        __syncthreads();
        if (kval) {
            const int t1 = t + 1, t2 = t + CTX, t3 = t + CTX + 1;   // cells 10, 01, 11 of the corner
            const double dzim = a.mz.dim[s - 1];
            double un[8];
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const double u0 = pu(L, par, q, t), u1 = pu(L, par, q, t1), u2 = pu(L, par, q, t2), u3 = pu(L, par, q, t3);
                const double uh = (uhp[q] + u1 + u0 + u3 + u2) / 8.0;
                uhp[q] = u1 + u0 + u3 + u2;
                double dfdx = 0.0, dfdy = 0.0, dfdz = 0.0;
                if (q != 5) {
                    const double f0 = px(L, par, q, t), f1 = px(L, par, q, t1), f2 = px(L, par, q, t2), f3 = px(L, par, q, t3);
                    dfdx = (fxp[q] + f1 - f0 + f3 - f2) / 4.0 * dxim;
                    fxp[q] = f1 - f0 + f3 - f2;
                }
                if (q != 6) {
                    const double f0 = py(L, q, t), f1 = py(L, q, t1), f2 = py(L, q, t2), f3 = py(L, q, t3);
                    dfdy = (fyp[q] + f2 - f0 + f3 - f1) / 4.0 * dyim;
                    fyp[q] = f2 - f0 + f3 - f1;
                }
                if (q != 7)
                    dfdz = (pz(L, par, q, t) - pz(L, lp, q, t) + pz(L, par, q, t1) - pz(L, lp, q, t1)
                            + pz(L, par, q, t2) - pz(L, lp, q, t2) + pz(L, par, q, t3) - pz(L, lp, q, t3)) / 4.0 * dzim;
                un[q] = uh - dt * dfdx - dt * dfdy - dt * dfdz;
                if (kSrc[q] >= 0) {   // mlwsrch.f:39-46
                    const int e = L_SRC + kSrc[q];
                    const double c0 = L.c[e][t], c1 = L.c[e][t1], c2 = L.c[e][t2], c3 = L.c[e][t3];
                    const double sh = (shp[kSrc[q]] + c1 + c0 + c3 + c2) / 8.0;
                    shp[kSrc[q]] = c1 + c0 + c3 + c2;
                    un[q] = un[q] + dt * sh;
                }
            }
            State h;
            h.ro = un[0]; h.bx = un[5]; h.by = un[6]; h.bz = un[7];
            h.vx = un[2] / h.ro;
            h.vy = un[3] / h.ro;
            h.vz = un[4] / h.ro;
            const double vv = h.vx * h.vx + h.vy * h.vy + h.vz * h.vz;
            const double bb = h.bx * h.bx + h.by * h.by + h.bz * h.bz;
            h.pr = (gm - 1.0) * (un[1] - 0.5 * h.ro * vv - pi8i * bb);
            Vals f;
            vals_x(h, gm, f);
            vals_y(h, gm, rm, f);
            vals_z(h, gm, f);
            vals_src(h, rm, p4rm, p8rm, f);
            double *o = a.corner + sz * (s - 1);   // at the index of cell (i, j, k)
#define W(slot, v) st(o + (size_t)(slot) * N, boff, v)
            W(Z_ROX, f.rox); W(Z_EEX, f.eex); W(Z_RXX, f.rxx); W(Z_RYX, f.ryx); W(Z_RZX, f.rzx);
            W(Z_EX, f.ex); W(Z_EY, f.ey); W(Z_EZ, f.ez);
            W(Z_FRO, f.fro); W(Z_FEE, f.fee); W(Z_FRX, f.frx); W(Z_FRY, f.fry); W(Z_FRZ, f.frz);
            W(Z_FBX, f.fbx); W(Z_FBZ, f.fbz);
            W(Z_ROZ, f.roz); W(Z_EEZ, f.eez); W(Z_RXZ, f.rxz); W(Z_RYZ, f.ryz); W(Z_RZZ, f.rzz);
#pragma unroll
            for (int q = 0; q < 6; q++) W(Z_SRO + q, f.src[q]);
#undef W
        }
        __syncthreads();   // the next plane's values replace these
    }
}

// corner flux of equation q at p
CANS_DEV double hx_(const double *h, size_t N, int q, size_t p) {
    switch (q) {
    case 5: return 0.0;
    case 6: return -h[Z_EZ * N + p];
    case 7: return h[Z_EY * N + p];
    default: return h[(size_t)(Z_ROX + q) * N + p];
    }
}
CANS_DEV double hy_(const double *h, size_t N, int q, size_t p) {
    return q == 6 ? 0.0 : h[(size_t)(Z_FRO + (q == 7 ? 6 : q)) * N + p];
}
CANS_DEV double hz_(const double *h, size_t N, int q, size_t p) {
    switch (q) {
    case 5: return -h[Z_EY * N + p];
    case 6: return h[Z_EX * N + p];
    case 7: return 0.0;
    default: return h[(size_t)(Z_ROZ + q) * N + p];
    }
}
CANS_DEV State load_state(const Mlw3dArgs &a, size_t p) {
    return State{a.prim[0][p], a.prim[1][p], a.prim[2][p], a.prim[3][p],
                 a.prim[4][p], a.prim[5][p], a.prim[6][p], a.prim[7][p]};
}

// interior cell (i,j,k) in [2,n-1]^3
__global__ __launch_bounds__(256) void cyl_update(Mlw3dArgs a) {
    double dt;
    if (!cyl_dt(a, dt)) return;
    const int ix = a.ix, jx = a.jx, kx = a.kx;
    const int ni = ix - 2, nj = jx - 2, nk = kx - 2;
    const size_t t = xcd_first_thread() + threadIdx.x;
    if (t >= (size_t)ni * nj * nk) return;
    const int i = 2 + (int)(t % ni);
    const int j = 2 + (int)((t / ni) % nj);
    const int k = 2 + (int)(t / ((size_t)ni * nj));
    const size_t N = (size_t)ix * jx * kx;
    const size_t sx = 1, sy = ix, sz = (size_t)ix * jx;
    const size_t p = (size_t)(i - 1) + sy * (j - 1) + sz * (k - 1);
    const double *h = a.corner;
    const double gm = a.gm, zero = 0.0;
    const double dxi = a.mx.di[i - 1], dyi = a.my.di[j - 1], dzi = a.mz.di[k - 1];
    const double dxim = a.mx.dim[i - 1], dyim = a.my.dim[j - 1], dzim = a.mz.dim[k - 1];
    const double dxim1 = a.mx.dim[i - 2], dyim1 = a.my.dim[j - 2], dzim1 = a.mz.dim[k - 2];
    const double ux0 = a.mx.u0[i - 1], ux1 = a.mx.u1[i - 1];
    const double uy0 = a.my.u0[j - 1], uy1 = a.my.u1[j - 1];
    const double uz0 = a.mz.u0[k - 1], uz1 = a.mz.u1[k - 1];
    const double r = a.x[i - 1];
    // centre terms of mlwhalf and the terms of mlwartv, axis by axis
    double U[8], du[8], ax[8], ay[8], az[8];
    const State C = load_state(a, p);
    conserved(C, gm, U);
    {
        const State E = load_state(a, p + sx), W = load_state(a, p - sx);
        double uE[8], uW[8];
        Vals fE, fW;
        conserved(E, gm, uE);
        conserved(W, gm, uW);
        vals_x(E, gm, fE);
        vals_x(W, gm, fW);
        const double qe = a.qav * a.dxm[i - 1] * fmaxF(zero, __builtin_fabs(E.vx - C.vx) - kR4_1em4);
        const double qw = a.qav * a.dxm[i - 2] * fmaxF(zero, __builtin_fabs(C.vx - W.vx) - kR4_1em4);
#pragma unroll
        for (int q = 0; q < 8; q++) {
            du[q] = 0.0;
            du[q] = du[q] - 0.5 * dt * (0.5 * dxi * (xflux(fE, q) - xflux(fW, q)));
            ax[q] = dt * (dxi * (qe * dxim * (uE[q] - U[q]) - qw * dxim1 * (U[q] - uW[q])));
        }
    }
    {
        const State E = load_state(a, p + sy), W = load_state(a, p - sy);
        double uE[8], uW[8];
        Vals fE, fW;
        conserved(E, gm, uE);
        conserved(W, gm, uW);
        vals_y(E, gm, r, fE);
        vals_y(W, gm, r, fW);
        const double qe = a.qav * a.dym[j - 1] * fmaxF(zero, __builtin_fabs(E.vy - C.vy) - kR4_1em4);
        const double qw = a.qav * a.dym[j - 2] * fmaxF(zero, __builtin_fabs(C.vy - W.vy) - kR4_1em4);
#pragma unroll
        for (int q = 0; q < 8; q++) {
            du[q] = du[q] - 0.5 * dt * (0.5 * dyi * (yflux(fE, q) - yflux(fW, q)));
            ay[q] = dt * (dyi * (qe * dyim * (uE[q] - U[q]) - qw * dyim1 * (U[q] - uW[q])));
        }
    }
    {
        const State E = load_state(a, p + sz), W = load_state(a, p - sz);
        double uE[8], uW[8];
        Vals fE, fW;
        conserved(E, gm, uE);
        conserved(W, gm, uW);
        vals_z(E, gm, fE);
        vals_z(W, gm, fW);
        const double qe = a.qav * a.dzm[k - 1] * fmaxF(zero, __builtin_fabs(E.vz - C.vz) - kR4_1em4);
        const double qw = a.qav * a.dzm[k - 2] * fmaxF(zero, __builtin_fabs(C.vz - W.vz) - kR4_1em4);
#pragma unroll
        for (int q = 0; q < 8; q++) {
            du[q] = du[q] - 0.5 * dt * (0.5 * dzi * (zflux(fE, q) - zflux(fW, q)));
            az[q] = dt * (dzi * (qe * dzim * (uE[q] - U[q]) - qw * dzim1 * (U[q] - uW[q])));
        }
    }
    {
        Vals f;
        vals_x(C, gm, f);
        vals_src(C, r, pi4i / r, 2.0 * pi4i / r, f);
#pragma unroll
        for (int q = 0; q < 8; q++)
            if (kSrc[q] >= 0) du[q] = du[q] + 0.5 * dt * f.src[kSrc[q]];   // mlwsrch.f:33-38
    }
    // corners around the cell: (i-1|i, j-1|j, k-1|k)
    const size_t c000 = p - sx - sy - sz;
    const size_t c100 = c000 + sx, c010 = c000 + sy, c110 = c010 + sx;
    const size_t c001 = c000 + sz, c101 = c001 + sx, c011 = c001 + sy, c111 = c011 + sx;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        // mlwfull
        const double dfdx = dxi * (uz0 * (uy0 * (hx_(h, N, q, c100) - hx_(h, N, q, c000))
                                          + uy1 * (hx_(h, N, q, c110) - hx_(h, N, q, c010)))
                                   + uz1 * (uy0 * (hx_(h, N, q, c101) - hx_(h, N, q, c001))
                                            + uy1 * (hx_(h, N, q, c111) - hx_(h, N, q, c011))));
        const double dfdy = dyi * (ux0 * (uz0 * (hy_(h, N, q, c010) - hy_(h, N, q, c000))
                                          + uz1 * (hy_(h, N, q, c011) - hy_(h, N, q, c001)))
                                   + ux1 * (uz0 * (hy_(h, N, q, c110) - hy_(h, N, q, c100))
                                            + uz1 * (hy_(h, N, q, c111) - hy_(h, N, q, c101))));
        const double dfdz = dzi * (uy0 * (ux0 * (hz_(h, N, q, c001) - hz_(h, N, q, c000))
                                          + ux1 * (hz_(h, N, q, c101) - hz_(h, N, q, c100)))
                                   + uy1 * (ux0 * (hz_(h, N, q, c011) - hz_(h, N, q, c010))
                                            + ux1 * (hz_(h, N, q, c111) - hz_(h, N, q, c110))));
        du[q] = du[q] - 0.5 * dt * dfdx - 0.5 * dt * dfdy - 0.5 * dt * dfdz;
        if (kSrc[q] >= 0) {   // mlwsrcf.f:33-46
            const double *sh_ = h + (size_t)(Z_SRO + kSrc[q]) * N;
            const double sh = uz0 * (uy0 * (ux0 * sh_[c000] + ux1 * sh_[c100]) + uy1 * (ux0 * sh_[c010] + ux1 * sh_[c110]))
                              + uz1 * (uy0 * (ux0 * sh_[c001] + ux1 * sh_[c101])
                                       + uy1 * (ux0 * sh_[c011] + ux1 * sh_[c111]));
            du[q] = du[q] + 0.5 * dt * sh;
        }
        du[q] = du[q] + ax[q] + ay[q] + az[q];
        U[q] = U[q] + du[q];
    }
    const double ro = U[0];
    const double vx = U[2] / ro;
    const double vy = U[3] / ro;
    const double vz = U[4] / ro;
    const double vv = vx * vx + vy * vy + vz * vz;
    const double bb = U[5] * U[5] + U[6] * U[6] + U[7] * U[7];
    a.out[0][p] = ro;
    a.out[1][p] = (gm - 1.0) * (U[1] - 0.5 * ro * vv - pi8i * bb);
    a.out[2][p] = vx;
    a.out[3][p] = vy;
    a.out[4][p] = vz;
    a.out[5][p] = U[5];
    a.out[6][p] = U[6];
    a.out[7][p] = U[7];
}

}  // namespace

hipError_t launch_mlw3d_cyl(const Mlw3dArgs &a, hipStream_t s) {
    if (a.ix < 3 || a.jx < 3 || a.kx < 3) return hipSuccess;
    if (!a.xm) return hipErrorInvalidValue;
    // The tile shape and the z-segments: a block is alone on its CU (its LDS),
    // so a launch takes rounds of 256; the number of segments with the fewest
    // planes per CU, one plane read before a segment's first corner, and the
    // shape that needs the fewest then, the widest of equal ones.  Narrow grids
    // leave most lanes of a wide tile idle: 7 x 189 x 260 cells, a step 489 us
    // with 64 x 8 tiles, 131 with 8 x 64 (175 with the three kernels).  A plane
    // of a narrow tile that is a piece of its rows takes a third longer (8 or 16
    // cells in a row of memory): 202 x 126 x 187, 56 planes of 64 x 8 tiles 1162
    // us a step, 48 of 8 x 64 1217; 65 x 31 x 158, 8 planes 121, 5 of 16 x 32 113.
    const int nz = a.kx - 1;
    int ctx = 0, wx = 0, wy = 0, tiles_x = 0, ntiles = 0, nseg = 1;
    long best = -1;
    for (int c : {64, 16, 8}) {
        const int mx = c - 1, my = CNT / c - 1;             // corners of a tile
        const int tx = (a.ix - 1 + mx - 1) / mx, ty = (a.jx - 1 + my - 1) / my;
        for (int n = 1; n <= 256 && n <= nz; n++) {
            const int len = (nz + n - 1) / n;
            const int used = (nz + len - 1) / len;
            const long cost = (((long)tx * ty * used + 256 - 1) / 256) * (len + 1) * (c < 64 && tx > 1 ? 4 : 3);
            if (best >= 0 && cost >= best) continue;
            best = cost;
            ctx = c; tiles_x = tx; ntiles = tx * ty; nseg = used;
            wx = (a.ix - 1 + tx - 1) / tx; wy = (a.jx - 1 + ty - 1) / ty;
        }
    }
    const int seglen = (nz + nseg - 1) / nseg;
    const long items = (long)ntiles * nseg;
    const unsigned grid = (unsigned)((items + kXcds - 1) / kXcds * kXcds);
#define CORNERS(c) hipLaunchKernelGGL(cyl_corners<c>, dim3(grid), dim3(CNT), 0, s, a, wx, wy, tiles_x, ntiles, nseg, seglen)
    if (ctx == 64) CORNERS(64);
    else if (ctx == 16) CORNERS(16);
    else CORNERS(8);
#undef CORNERS
    if (hipError_t e = hipGetLastError()) return e;
    const size_t nu = (size_t)(a.ix - 2) * (a.jx - 2) * (a.kx - 2);
    hipLaunchKernelGGL(cyl_update, dim3(xcd_grid(nu)), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace cans

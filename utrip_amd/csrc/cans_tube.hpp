// cans_tube.hpp -- the 1D modified Lax-Wendroff update (cans1d/hdmlw/mlw_m.f:
// 2-215) of one cell per lane, neighbours by DPP lane shifts: the row code of
// the batched tubes and of the resident 1D run.
#pragma once
#include "cans_common.hpp"
#include "cans_wave.hpp"

namespace cans {

struct Tube {
    double ro, pr, vx, vy, by;
};

// The updated cell of this lane from its primitives w, bx, bxm and metric
// (di = 1/dx, dim = 1/dxm); valid in lanes 1..62, whose neighbours are the
// adjacent lanes.  T = double: mlw_m bit for bit; T = float: cell and face
// fluxes (and their differences) in FP32, the rest FP64.
template <class T>
CANS_DEV Tube tube_update(const Tube &w, double bx, double bxm, double dxi, double dxim, double dxm, double dt,
                          double qav, double gm) {
    constexpr double pi8i = 1.0 / kPi / 8.0;   // mlw_m.f:55
    constexpr double pi4i = 1.0 / kPi / 4.0;   // mlw_m.f:56
    const double ro = w.ro, pr = w.pr, vx = w.vx, vy = w.vy, by = w.by;
    // cells (mlw_m.f:79-125): conserved variables in FP64, fluxes in T
    double u[5];
    T f[5];
    {
        const double vv = vx * vx + vy * vy;
        const double bb = by * by;
        u[0] = ro;
        u[1] = pr / (gm - 1.0) + 0.5 * ro * vv + pi8i * bb;
        u[2] = ro * vx;
        u[3] = ro * vy;
        u[4] = by;
        const T tro = (T)ro, tpr = (T)pr, tvx = (T)vx, tvy = (T)vy, tby = (T)by, tbx = (T)bx, tgm = (T)gm;
        const T tvv = tvx * tvx + tvy * tvy;
        const T tbb = tby * tby;
        const T ez = -tvx * tby + tvy * tbx;
        const T ep = tpr * tgm / (tgm - (T)1.0) + (T)0.5 * tro * tvv;
        f[0] = tro * tvx;
        f[1] = ep * tvx - tby * ez * (T)pi4i;
        f[2] = tro * (tvx * tvx) + tpr + tbb * (T)pi8i;
        f[3] = tro * tvx * tvy - tbx * tby * (T)pi4i;
        f[4] = -ez;
    }
    // face between this cell and the next (mlwhalf.f:39-46, mlw_m.f:129-175):
    // the half-step state and its primitives, pressure included, in FP64
    // (in the mixed form the flux difference that enters it is the FP32 one,
    // widened); the face fluxes in T.
    T ff[5];
    T fE[5];
    double uE[5];
    {
        double un[5];
#pragma unroll
        for (int q = 0; q < 5; q++) {
            uE[q] = shl1(u[q]);
            fE[q] = shl1(f[q]);
            const double uh = 0.5 * (uE[q] + u[q]);
            const double dfdx = dxim * (double)(fE[q] - f[q]);
            un[q] = uh - dt * dfdx;
        }
        const double roh = un[0], eeh = un[1], rxh = un[2], ryh = un[3], byh = un[4];
        const double vxh = rxh / roh;
        const double vyh = ryh / roh;
        const double vv = vxh * vxh + vyh * vyh;
        const double bb = byh * byh;
        const double prh = (gm - 1.0) * (eeh - 0.5 * roh * vv - pi8i * bb);
        const T troh = (T)roh, tvxh = (T)vxh, tvyh = (T)vyh, tbyh = (T)byh, tbxm = (T)bxm, tprh = (T)prh,
                tgm = (T)gm;
        const T tvv = tvxh * tvxh + tvyh * tvyh;
        const T tbb = tbyh * tbyh;
        const T ezh = -tvxh * tbyh + tvyh * tbxm;
        const T eph = tprh * tgm / (tgm - (T)1.0) + (T)0.5 * troh * tvv;
        ff[0] = troh * tvxh;
        ff[1] = eph * tvxh - tbyh * ezh * (T)pi4i;
        ff[2] = troh * (tvxh * tvxh) + tprh + tbb * (T)pi8i;
        ff[3] = troh * tvxh * tvyh - tbxm * tbyh * (T)pi4i;
        ff[4] = -ezh;
    }
    // own cell: centre term, full step, artificial viscosity, update
    const double zero = 0.0;
    const double vxE = shl1(vx);
    const double qxc = qav * dxm * fmaxF(zero, __builtin_fabs(vxE - vx) - kR4_1em4);
    const double qxw = shr1(qxc);            // qav*dxm(c-1)*max(0,|vx(c)-vx(c-1)|-1e-4)
    const double dxim1 = shr1(dxim);
    double du[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {
        du[q] = 0.0;
        const T fW = shr1(f[q]);
        du[q] = du[q] - 0.5 * dt * (0.5 * dxi * (double)(fE[q] - fW));      // mlwhalf.f:33-35
        const T dfdx = (T)dxi * (ff[q] - shr1(ff[q]));                      // mlwfull.f:30-33
        du[q] = du[q] - 0.5 * dt * (double)dfdx;
        const double dEc = uE[q] - u[q];                                    // mlwartv.f:31-34
        const double dcW = shr1(dEc);
        du[q] = du[q] + dt * (dxi * (qxc * dxim * dEc - qxw * dxim1 * dcW));
    }
    const double nro = u[0] + du[0];
    const double nrx = u[2] + du[2];
    const double nry = u[3] + du[3];
    const double nby = u[4] + du[4];
    const double nee = u[1] + du[1];
    const double nvx = nrx / nro;
    const double nvy = nry / nro;
    const double nvv = nvx * nvx + nvy * nvy;
    const double nbb = nby * nby;
    const double npr = (gm - 1.0) * (nee - 0.5 * nro * nvv - pi8i * nbb);
    return Tube{nro, npr, nvx, nvy, nby};
}

}  // namespace cans

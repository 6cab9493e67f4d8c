// cans_run1d.hip -- many steps of one resident 1D run in one launch: the
// CANS loop {cfl_m; stop on merr; t = t+dt; mlw_m; bnd} of
// cans1d/md_mhdshktb/hdmlw/main.f:132-186 for a tube whose faces copy
// interior cells (BndMap: bdfrex, bdspp/spnx, bdsmpx, bdperx).
//
// A 1D tube is a few thousand cells: a step of it is a microsecond or two of
// one CU, and a launch per routine (cfl_m, clock, engine, a fill per face)
// costs ten times that.  One workgroup therefore keeps the tube and runs its
// steps back to back: waves update 62-cell segments (tube_update, the row
// code of the batched tubes), the cell at a face writes its ghost copies, the
// next step's cfl_m term is taken with the update, and the step's only
// barrier is the dt minimum.  What bounds it is one CU's FP64 issue (about
// 480 instructions per segment; 1024 cells, 17 segments on 4 SIMDs: 82 % of
// the step's 4.4 us) and, up to a segment a SIMD, the step's one chain of
// dependent FP64 operations (2.0 us).  Measured, us a step, against the
// launches: 256 cells 15.3 -> 2.7, 1024 16.6 -> 4.4, 2000 16.7 -> 7.4, 4000
// 17.1 -> 14.1.
// The two buffers of the state live in LDS, with the six per-cell
// coefficients beside them while they fit (kCapAll cells), then without
// (kCapState), so that a step waits on no memory; longer tubes keep the
// buffers in memory, through the CU's own L1 and its L2.
#include "cans_common.hpp"
#include "cans_clock.hpp"
#include "cans_kernels.hpp"
#include "cans_tube.hpp"
#include "cans_wave.hpp"

namespace cans {
namespace {

enum { LDS_ALL, LDS_STATE, LDS_NONE };
constexpr int kCapAll = 1264;     // 2*5 + 6 doubles a cell in 160 KB
constexpr int kCapState = 2032;   // 2*5 doubles a cell
enum { K_BX, K_BXM, K_DX, K_DXM, K_DI, K_DIM, K_N };

template <int MODE>
struct TubeMem {
    static constexpr int cap = MODE == LDS_ALL ? kCapAll : (MODE == LDS_STATE ? kCapState : 1);
    double s[2][5][cap];
    double k[MODE == LDS_ALL ? K_N : 1][MODE == LDS_ALL ? cap : 1];
};

// ghost cells that copy cell c: count and first, per side (Images of the 2D
// kernel, for the one axis)
struct Ghosts {
    int n, t;
};
CANS_DEV Ghosts ghosts_of(const Run1dArgs &a, int side, int c) {
    const int n = a.ix, m = a.margin, e = n - m, k = a.kind[side];
    if (side == 0) {
        if (k == BM_FRE) return Ghosts{c == m + 1 ? m : 0, 1};
        if (k == BM_SP) return Ghosts{c >= m + 1 && c <= 2 * m, 2 * m + 1 - c};
        if (k == BM_SM) return Ghosts{c >= m + 2 && c <= 2 * m + 1, 2 * m + 2 - c};
        return Ghosts{c >= n - 2 * m + 1 && c <= e, c - (n - 2 * m)};
    }
    if (k == BM_FRE) return Ghosts{c == e ? m : 0, e + 1};
    if (k == BM_SP) return Ghosts{c >= e - m + 1 && c <= e, 2 * e + 1 - c};
    if (k == BM_SM) return Ghosts{c >= e - m && c <= e - 1, 2 * e - c};
    return Ghosts{c >= m + 1 && c <= 2 * m, c + (n - 2 * m)};
}

template <int BT, int MODE>
__global__ __launch_bounds__(BT) void run1d_kernel(Run1dArgs a) {
    constexpr int NW = BT / 64;
    __shared__ TubeMem<MODE> M;
    __shared__ double red[2][NW];
    const int ix = a.ix, margin = a.margin;
    const int lane = threadIdx.x & 63;
    const int wv = uni((int)(threadIdx.x >> 6));
    // the state of step0: set a for an even step, b for an odd one; step n
    // writes the other
    double *const *in = (a.step0 & 1) ? a.b : a.a;
    const double *kg[K_N] = {a.bx, a.bxm, a.dx, a.dxm, a.di, a.dim};
    if (MODE != LDS_NONE) {
        for (int p = (int)threadIdx.x; p < ix; p += BT) {
#pragma unroll
            for (int q = 0; q < 5; q++) M.s[0][q][p] = in[q][p];
            if (MODE == LDS_ALL) {
#pragma unroll
                for (int q = 0; q < K_N; q++) M.k[q][p] = kg[q][p];
            }
        }
        __syncthreads();
    }
    auto coef = [&](int q, int p) { return MODE == LDS_ALL ? M.k[q][p] : kg[q][p]; };

    // the clock of the step (clock_enter's control flow, kept in scalars)
    Clock *clk = a.clk;
    const int sl = a.step0 & 1;
    double t = uni(clk->t[sl]), dt_last = uni(clk->dt_last[sl]);
    int ns = uni(clk->ns[sl]), nexec = uni(clk->nexec[sl]), merr = uni(clk->merr[sl]), stopped = uni(clk->stopped[sl]);
    const double tend = uni(clk->tend), dtmin = uni(clk->dtmin);
    const int nstop = uni(clk->nstop);

    // cfl_m of the state the call finds, over i = 2..ix-1
    double m = kR4_1e20;
    for (int c = 2 + (int)threadIdx.x; c <= ix - 1; c += BT) {
        const int p = c - 1;
        double w[5];
#pragma unroll
        for (int q = 0; q < 5; q++) w[q] = MODE == LDS_NONE ? in[q][p] : M.s[0][q][p];
        const double d = dtq1(w[0], w[1], w[2], w[4], coef(K_BX, p), coef(K_DX, p), a.gm, a.safety);
        if (d < m) m = d;
    }
    int par = 0;
    double dt = block_min<BT>(m, red[par]);
    par ^= 1;
    const int nseg = (ix - 2 * margin + 61) / 62;
    int done = 0;                                  // steps this call executed
    for (int n = 0; n < a.nsteps; n++) {
        if (stopped || !(ns < nstop && t < tend)) { stopped = 1; break; }
        ns = ns + 1;
        if (dt < dtmin) { merr = 9001; stopped = 1; break; }   // cfl_m.f: merr=9001
        t = t + dt;
        dt_last = dt;
        const int cur = done & 1, nxt = cur ^ 1;
        double *const *gc = ((a.step0 + done) & 1) ? a.b : a.a;
        double *const *gn = ((a.step0 + done) & 1) ? a.a : a.b;
        m = kR4_1e20;
        for (int s = wv; s < nseg; s += NW) {
            const int c = margin + 62 * s + lane;                 // 1-based; lane 0 is the west halo
            const int p = (c < 1 ? 1 : (c > ix ? ix : c)) - 1;
            double w[5];
#pragma unroll
            for (int q = 0; q < 5; q++) w[q] = MODE == LDS_NONE ? gc[q][p] : M.s[cur][q][p];
            const double bx = coef(K_BX, p);
            const Tube u = tube_update<double>(Tube{w[0], w[1], w[2], w[3], w[4]}, bx, coef(K_BXM, p), coef(K_DI, p),
                                               coef(K_DIM, p), coef(K_DXM, p), dt, a.qav, a.gm);
            if (lane >= 1 && lane <= 62 && c <= ix - margin) {
                const double o[5] = {u.ro, u.pr, u.vx, u.vy, u.by};
#pragma unroll
                for (int q = 0; q < 5; q++) (MODE == LDS_NONE ? gn[q][p] : M.s[nxt][q][p]) = o[q];
                if (c >= 2 && c <= ix - 1) {
                    const double d = dtq1(u.ro, u.pr, u.vx, u.by, bx, coef(K_DX, p), a.gm, a.safety);
                    if (d < m) m = d;
                }
                if (c <= 2 * margin + 1 || c >= ix - 2 * margin) {
                    for (int side = 0; side < 2; side++) {
                        const Ghosts g = ghosts_of(a, side, c);
                        for (int k = 0; k < g.n; k++) {
                            const int pg = g.t + k - 1;
#pragma unroll
                            for (int q = 0; q < 5; q++)
                                (MODE == LDS_NONE ? gn[q][pg] : M.s[nxt][q][pg]) = (a.neg[side] >> q) & 1u ? -o[q] : o[q];
                            if (pg >= 1 && pg <= ix - 2) {        // cfl_m sees cells 2..ix-1
                                const double d = dtq1(u.ro, u.pr, u.vx, u.by, coef(K_BX, pg), coef(K_DX, pg), a.gm,
                                                      a.safety);
                                if (d < m) m = d;
                            }
                        }
                    }
                }
            }
        }
        done++;
        dt = block_min<BT>(m, red[par]);           // dt of the next step; also the step's barrier
        par ^= 1;
    }
    // the last two states back to their buffer sets (the first of them only
    // if a step of this call made it)
    if (MODE != LDS_NONE) {
        for (int back = 0; back < 2 && back < done; back++) {
            double *const *dst = ((a.step0 + done - back) & 1) ? a.b : a.a;
            const int from = (done - back) & 1;
            for (int p = (int)threadIdx.x; p < ix; p += BT) {
#pragma unroll
                for (int q = 0; q < 5; q++) dst[q][p] = M.s[from][q][p];
            }
        }
    }
    if (wv == 0) {   // uniform branch; the lanes store identical values
#pragma unroll
        for (int s = 0; s < 2; s++) {
            clk->t[s] = t;
            clk->dt_last[s] = dt_last;
            clk->ns[s] = ns;
            clk->nexec[s] = nexec + done;
            clk->merr[s] = merr;
            clk->stopped[s] = stopped;
        }
#pragma unroll
        for (int s = 0; s < 3; s++) clk->dtkey[s] = dkey(kR4_1e20);
    }
}

}  // namespace

hipError_t launch_run1d(const Run1dArgs &a, hipStream_t s) {
    const int nseg = (a.ix - 2 * a.margin + 61) / 62;   // a wave per segment while there are waves
    if (a.ix > kCapState) hipLaunchKernelGGL((run1d_kernel<1024, LDS_NONE>), dim3(1), dim3(1024), 0, s, a);
    else if (a.ix > kCapAll) hipLaunchKernelGGL((run1d_kernel<1024, LDS_STATE>), dim3(1), dim3(1024), 0, s, a);
    else if (nseg > 8) hipLaunchKernelGGL((run1d_kernel<1024, LDS_ALL>), dim3(1), dim3(1024), 0, s, a);
    else if (nseg > 4) hipLaunchKernelGGL((run1d_kernel<512, LDS_ALL>), dim3(1), dim3(512), 0, s, a);
    else hipLaunchKernelGGL((run1d_kernel<256, LDS_ALL>), dim3(1), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace cans

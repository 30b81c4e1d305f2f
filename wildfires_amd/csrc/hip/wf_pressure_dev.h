/*
 * wf_pressure_dev.h -- device functions shared by the two forms of the
 * pressure solve: the Poisson right-hand side at a node, the convergence check
 * of the fixed-point iteration, and the operands of a batched member.
 */
#ifndef WF_PRESSURE_DEV_H
#define WF_PRESSURE_DEV_H

#include "wf_common.h"
#include "wf_kernels.h"

#define WF_NT 256 /* threads of the x- and y-transform workgroups and of the check */

namespace WF_NS {

__device__ __forceinline__ wf_real2 wf_make2(wf_real x, wf_real y) {
    wf_real2 r;
    r.x = x;
    r.y = y;
    return r;
}

/* 32-bit element offsets from a uniform base (scalar base + 32-bit lane offset;
 * the solver limits Nx*Ny*Nz to 2^28). */
__device__ __forceinline__ wf_real wf_ldp(const wf_real *base, unsigned q) {
    return *(const wf_real *)((const char *)base + q * (unsigned)sizeof(wf_real));
}

/* v of another lane of the row of 16 (or of the rows before), by DPP control
 * CTRL; lanes without a source keep v. */
template <int CTRL>
__device__ __forceinline__ double wf_dpp(double v) {
    const int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false),
                            __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false));
}
__device__ __forceinline__ double wf_max2(double a, double b) { return (b > a) ? b : a; }
/* Maximum of v over the wavefront, in lane 63 (swaps within 16 lanes, then
 * the row broadcasts): vector instructions, where the shuffles go through LDS
 * and cost a microsecond of every pass's end. */
__device__ __forceinline__ double wf_wave_max(double v) {
    v = wf_max2(v, wf_dpp<0xb1>(v));  /* quad_perm 1 0 3 2 */
    v = wf_max2(v, wf_dpp<0x4e>(v));  /* quad_perm 2 3 0 1 */
    v = wf_max2(v, wf_dpp<0x141>(v)); /* row_half_mirror */
    v = wf_max2(v, wf_dpp<0x140>(v)); /* row_mirror */
    v = wf_max2(v, wf_dpp<0x142>(v)); /* row_bcast 15 */
    v = wf_max2(v, wf_dpp<0x143>(v)); /* row_bcast 31 */
    return v;
}
/* Maximum of v over the workgroup, written by thread 0 to *out. */
__device__ __forceinline__ void wf_block_max_store(double v, double *out) {
    __shared__ double red[16];
    v = wf_wave_max(v);
    if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = red[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) m = (red[w] > m) ? red[w] : m;
        *out = m;
    }
}

/* p-independent part of f at node (i,j,k), 1 <= k <= Nz-2
 * (src/cu/pressure.cu:14-101 for constant density, 103-327 otherwise).
 * [Q1] h_c per node with |T_gas - T_solid|. */
__device__ wf_real wf_f_fixed(const WfConst &c, const WfState &Ys, const WfState &Yn, int i, int j, int k) {
    const int Nx = c.Nx, Ny = c.Ny;
    const long P = c.plane;
    const wf_real *z = c.z;
    int im1 = wf_wrap_m(i, 1, Nx), ip1 = wf_wrap_p(i, 1, Nx);
    int jm1 = wf_wrap_m(j, 1, Ny), jp1 = wf_wrap_p(j, 1, Ny);
    long q = wf_q(c, i, j, k);
    long qxm = wf_q(c, im1, j, k), qxp = wf_q(c, ip1, j, k), qym = wf_q(c, i, jm1, k), qyp = wf_q(c, i, jp1, k);
    wf_real dz_km1 = z[k] - z[k - 1], dz_k = z[k + 1] - z[k];
    wf_real u = Ys.u[q], v = Ys.v[q];
    wf_real wz = (Ys.w[q + P] - Ys.w[q - P]) / (dz_k + dz_km1);
    wf_real u_iph = WR(0.5) * (Ys.u[qxp] + u), u_imh = WR(0.5) * (u + Ys.u[qxm]);
    wf_real v_jph = WR(0.5) * (Ys.v[qyp] + v), v_jmh = WR(0.5) * (v + Ys.v[qym]);
    wf_real ux = (u_iph - u_imh) / c.dx, vy = (v_jph - v_jmh) / c.dy;
    if (c.variable_density == 0) return c.rho_inf * (ux + vy + wz) / c.dt;
    wf_real T = Ys.T[q];
    wf_real Tip = Ys.T[qxp], Tim = Ys.T[qxm], Tjp = Ys.T[qyp], Tjm = Ys.T[qym];
    wf_real Tkp = Ys.T[q + P], Tkm = Ys.T[q - P];
    wf_real rho = c.T_inf * c.rho_inf / Yn.T[q];
    wf_real Tx = (Tip - Tim) / (2 * c.dx), Ty = (Tjp - Tjm) / (2 * c.dy);
    wf_real Txx = (Tip - 2 * T + Tim) / (c.dx * c.dx), Tyy = (Tjp - 2 * T + Tjm) / (c.dy * c.dy);
    wf_real Tz = (Tkp - Tkm) / (dz_k + dz_km1);
    wf_real Tzz = wf_d2m(Tkm, T, Tkp, dz_km1, dz_k);
    wf_real lap_T = Txx + Tyy + Tzz;
    wf_real kT = c.kT, dk = WR(0.0);
    wf_real Y = WR(0.0);
    wf_real K_T = wf_rate(c, T);
    wf_real T_gas = T, T_solid = T;
    int col = i + Nx * j;
    int nzy = c.nzy[col];
    if (k <= nzy) {
        if (k < nzy) Y = Ys.Y[q];
        if (Y > WR(0.0))
            T_gas = c.T_pc + (T - c.T_pc);
        else
            T_gas = T;
    }
    if (c.suth_k == 1) wf_sutherland_k(T, &kT, &dk);
    wf_real qs = c.H_C * Y * K_T / c.c_p;
    if (c.exchange_on) {
        wf_real h_c = c.h_c * dz_k * pow(fabs(T_gas - T_solid) / dz_k, WR(1.0) / WR(4.0));
        qs = qs - h_c * c.alpha_s * c.sigma_s * (T_gas - T_solid) / (c.c_p * c.T_inf * c.rho_inf / T_gas);
    }
    wf_real T2 = T * T, T3 = T * T * T;
    wf_real div_U_temp = (dk + 12 * WR(WF_SIGMA_D) * c.delta * T2 * (Tx * Tx + Ty * Ty + Tz * Tz) +
                         (kT + 4 * WR(WF_SIGMA_D) * c.delta * T3) * lap_T) / (c.T_inf * c.rho_inf * c.c_p) + qs / T;
    return rho * (ux + vy + wz - div_U_temp) / c.dt;
}

/* (grad rho . grad p) / rho at node (i,j,k), 1 <= k <= Nz-2, with rho = rho^n
 * the density of y_n (src/cu/pressure.cu:163-197, 269-282, 319).  The
 * constant divisors 2dx, 2dy, z[k+1]-z[k-1] are taken as reciprocals and the
 * sum divided by rho once. */
__device__ __forceinline__ wf_real wf_f_pgrad(const WfConst &c, const wf_real *rho_n, const wf_real *p, int i, int j,
                                             int k) {
#pragma clang fp contract(fast)
    const int Nx = c.Nx, Ny = c.Ny;
    const unsigned P = (unsigned)c.plane;
    const int im1 = wf_wrap_m(i, 1, Nx), ip1 = wf_wrap_p(i, 1, Nx);
    const int jm1 = wf_wrap_m(j, 1, Ny), jp1 = wf_wrap_p(j, 1, Ny);
    const unsigned q = (unsigned)wf_q(c, i, j, k);
    const unsigned qxm = (unsigned)wf_q(c, im1, j, k), qxp = (unsigned)wf_q(c, ip1, j, k);
    const unsigned qym = (unsigned)wf_q(c, i, jm1, k), qyp = (unsigned)wf_q(c, i, jp1, k);
    const wf_real dzc = c.zc[WF_ZC * k + WF_Z_DZC];
    const wf_real rho = wf_ldp(rho_n, q);
    const wf_real rhox = (wf_ldp(rho_n, qxp) - wf_ldp(rho_n, qxm)) * c.inv2dx;
    const wf_real rhoy = (wf_ldp(rho_n, qyp) - wf_ldp(rho_n, qym)) * c.inv2dy;
    const wf_real px = (wf_ldp(p, qxp) - wf_ldp(p, qxm)) * c.inv2dx;
    const wf_real py = (wf_ldp(p, qyp) - wf_ldp(p, qym)) * c.inv2dy;
    const wf_real rhoz = (wf_ldp(rho_n, q + P) - wf_ldp(rho_n, q - P)) * dzc;
    const wf_real pz = (wf_ldp(p, q + P) - wf_ldp(p, q - P)) * dzc;
    return (rhox * px + rhoy * py + rhoz * pz) / rho;
}

#if !WF_MIXED
/* v of the lane below (lane 0: edge) and of the lane above (lane 63: edge) */
__device__ __forceinline__ double wf_lane_below(double v, double edge) {
    return __hiloint2double(
        __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(v), 0x138, 0xf, 0xf, false),
        __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(v), 0x138, 0xf, 0xf, false));
}
__device__ __forceinline__ double wf_lane_above(double v, double edge) {
    return __hiloint2double(
        __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(v), 0x130, 0xf, 0xf, false),
        __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(v), 0x130, 0xf, 0xf, false));
}

/* The later iterations' input on the pair of nodes (i, ja), (i, ja + 1) of a
 * wavefront whose lanes hold consecutive columns i from a multiple of 64 on
 * (those past the last clamped to it) of one row pair: the two rows are each
 * other's y-neighbours (past the last row the second is row 0, and its result
 * of no meaning), the x-neighbours come from the lanes beside, except at the
 * ends of the wavefront and of the row. */
struct WfPairIn {
    wf_real A[2], a[2], b[2], ym[2], yp[2], azm[2], azp[2], bzm[2], bzp[2], ea[2], eb[2];
};
__device__ __forceinline__ void wf_pair_load(const WfConst &c, const wf_real *A, const wf_real *rho_n, const wf_real *p,
                                             int i, int ja, int k, WfPairIn &v) {
    const unsigned Nx = (unsigned)c.Nx, P = (unsigned)c.plane, zrow = (unsigned)c.Ny * (unsigned)k;
    const int jb = wf_wrap_p(ja, 1, c.Ny);
    const unsigned ra = Nx * (zrow + (unsigned)ja), rb = Nx * (zrow + (unsigned)jb);
    const unsigned rm = Nx * (zrow + (unsigned)wf_wrap_m(ja, 1, c.Ny)), rp = Nx * (zrow + (unsigned)wf_wrap_p(jb, 1, c.Ny));
    const int lane = (int)__lane_id();
    const unsigned ie = (unsigned)((lane == 0) ? wf_wrap_m(i, 1, c.Nx) : wf_wrap_p(i, 1, c.Nx));
    const wf_real *f[2] = {rho_n, p};
    v.A[0] = wf_ldp(A + ra, i);
    v.A[1] = wf_ldp(A + rb, i);
#pragma unroll
    for (int n = 0; n < 2; n++) {
        v.a[n] = wf_ldp(f[n] + ra, i);
        v.b[n] = wf_ldp(f[n] + rb, i);
        v.ym[n] = wf_ldp(f[n] + rm, i);
        v.yp[n] = wf_ldp(f[n] + rp, i);
        v.azm[n] = wf_ldp(f[n] + (ra - P), i);
        v.azp[n] = wf_ldp(f[n] + (ra + P), i);
        v.bzm[n] = wf_ldp(f[n] + (rb - P), i);
        v.bzp[n] = wf_ldp(f[n] + (rb + P), i);
        v.ea[n] = v.eb[n] = WR(0.0);
    }
    if (lane == 0 || lane == 63 || i >= c.Nx - 2) {
#pragma unroll
        for (int n = 0; n < 2; n++) {
            v.ea[n] = wf_ldp(f[n] + ra, ie);
            v.eb[n] = wf_ldp(f[n] + rb, ie);
        }
    }
}
/* wf_f_pgrad's operations, the contractions spelled out */
__device__ __forceinline__ void wf_pair_eval(const WfConst &c, const WfPairIn &v, int i, wf_real dzc, wf_real *fa,
                                             wf_real *fb) {
    const bool last = i >= c.Nx - 2;
    wf_real ax[2], ay[2], az[2], bx[2], by[2], bz[2];
#pragma unroll
    for (int n = 0; n < 2; n++) {
        const wf_real au = wf_lane_above(v.a[n], v.ea[n]), bu = wf_lane_above(v.b[n], v.eb[n]);
        ax[n] = ((last ? v.ea[n] : au) - wf_lane_below(v.a[n], v.ea[n])) * c.inv2dx;
        bx[n] = ((last ? v.eb[n] : bu) - wf_lane_below(v.b[n], v.eb[n])) * c.inv2dx;
        ay[n] = (v.b[n] - v.ym[n]) * c.inv2dy;
        by[n] = (v.yp[n] - v.a[n]) * c.inv2dy;
        az[n] = (v.azp[n] - v.azm[n]) * dzc;
        bz[n] = (v.bzp[n] - v.bzm[n]) * dzc;
    }
    *fa = v.A[0] + wf_fma(az[0], az[1], wf_fma(ay[0], ay[1], ax[0] * ax[1])) / v.a[0];
    *fb = v.A[1] + wf_fma(bz[0], bz[1], wf_fma(by[0], by[1], bx[0] * bx[1])) / v.b[0];
}
#endif

/* Maximum of the n partial maxima a[] (>= 0) over the workgroup, into *out
 * (16 independent loads per thread and pass, so one pass costs one memory
 * round trip; a plain strided loop waits for each load in turn). */
__device__ __forceinline__ void wf_reduce_max(const double *a, int n, double *out) {
    constexpr int U = 16;
    double v = 0.0;
    const int nt = (int)blockDim.x;
    for (int t0 = 0; t0 < n; t0 += U * nt) {
        double x[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int t = t0 + u * nt + (int)threadIdx.x;
            x[u] = (t < n) ? a[t] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; u++) v = (x[u] > v) ? x[u] : v;
    }
    wf_block_max_store(v, out);
    __syncthreads();
}

/* After solve m: err = max|p_new - p_old| (the maximum of the inverse
 * x-transform's per-workgroup maxima), stop once err <= tol or after max_iter
 * solves (src/cu/pressure.cu:564-574); iters is the count the reference
 * reports (the index of the converging solve, else max_iter).  The mixed form
 * also stops once err <= rtol max|p_new|: below that the FP32 iteration no
 * longer moves p toward the solution (its accuracy floor).  The flag and the
 * solve count are also written to mapped host memory so the host can stop
 * queueing solves without a round trip.
 *
 * The check of solve m is done by one extra workgroup (block 0) of solve
 * m + 1's first pass, beside the pass's own workgroups; only the last queued
 * solve is checked by a launch of its own (k_iter_check).  The pass's other
 * workgroups go on whether m converged or not (wf_iter.h).  As its own launch
 * after every solve the check took 4.3-6.2 us of latency, 5 % of a solve at
 * 256x256x128 and 12-17 % at 64x64x32 and below.  (Reducing in the inverse
 * transform itself would need a device-scope release, an L2 write-back, in
 * every workgroup.) */
__device__ __forceinline__ void wf_iter_check_body(const WfSpectral &sp, double tol, double rtol, int m,
                                                   int max_iter) {
    WfIterCtl *ctl = sp.ctl;
    if (wf_pass_returns(ctl->done)) return;
    __shared__ double err, pabs;
    wf_reduce_max(sp.pmax, sp.npmax, &err);
#if WF_MIXED
    wf_reduce_max(sp.pmax + sp.npmax, sp.npmax, &pabs);
#endif
    if (threadIdx.x != 0) return;
    double tol_eff = tol;
#if WF_MIXED
    tol_eff = (rtol * pabs > tol_eff) ? rtol * pabs : tol_eff;
#endif
    const int met = err <= tol_eff;
    const int iters = met ? m : m + 1, done = met || m + 1 >= max_iter;
    ctl->err = err;
    ctl->solves = m + 1;
    ctl->iters = iters;
    ctl->done = wf_iter_flag(done, m);
    volatile WfHostFlag *hf = sp.hflag;
    hf->err = err;
    hf->iters = iters;
    hf->solves = m + 1;
    if (!done) return;
    __threadfence_system();
    hf->done = 1;
    __threadfence_system();
}
/* Block index of a first pass whose block 0 checks the previous solve
 * (check >= 0: its index), -1 for that block after the check. */
__device__ __forceinline__ int wf_checked_block(const WfSpectral &sp, double tol, double rtol, int check,
                                                int max_iter) {
    if (check < 0) return (int)blockIdx.x;
    if (blockIdx.x == 0) wf_iter_check_body(sp, tol, rtol, check, max_iter);
    return (int)blockIdx.x - 1;
}

/* Input value of the x-transform at (i, j, k) for form MODE. */
template <int MODE>
__device__ __forceinline__ wf_real wf_fx_input(const WfConst &c, const WfSpectral &sp, const WfState &Ys,
                                              const WfState &Yn, const wf_real *p, int i, int j, int k) {
    long q = wf_q(c, i, j, k);
    if constexpr (MODE == WF_F_TOP) {
        return p[q];
    } else if constexpr (MODE == WF_F_CONST) {
        return wf_f_fixed(c, Ys, Yn, i, j, k);
    } else if constexpr (MODE == WF_F_FIRST) {
        wf_real f = wf_f_fixed(c, Ys, Yn, i, j, k);
        sp.A[q] = f;
        return f + wf_f_pgrad(c, sp.rho, p, i, j, k);
    } else {
        return sp.A[q] + wf_f_pgrad(c, sp.rho, p, i, j, k);
    }
}

/* member blockIdx.z's operands, every pointer global */
__device__ __forceinline__ WfPressItem wf_press_load(const WfPressItem *__restrict__ tab) {
    WfPressItem it = tab[blockIdx.z];
    wf_glob_const(it.c);
    WfSpectral &sp = it.sp;
    sp.F = wf_glob(sp.F);
    sp.Ptop = wf_glob(sp.Ptop);
    sp.A = wf_glob(sp.A);
    sp.UB = wf_glob(sp.UB);
    sp.pmax = wf_glob(sp.pmax);
    sp.kx2 = wf_glob(sp.kx2);
    sp.ky2 = wf_glob(sp.ky2);
    sp.ta = wf_glob(sp.ta);
    sp.tc = wf_glob(sp.tc);
    sp.kx2d = wf_glob(sp.kx2d);
    sp.ky2d = wf_glob(sp.ky2d);
    sp.tad = wf_glob(sp.tad);
    sp.tcd = wf_glob(sp.tcd);
    sp.betad = wf_glob(sp.betad);
    sp.twx = wf_glob(sp.twx);
    sp.twy = wf_glob(sp.twy);
    sp.radx = wf_glob(sp.radx);
    sp.rady = wf_glob(sp.rady);
    sp.beta = wf_glob(sp.beta);
    sp.rho = wf_glob(sp.rho);
    sp.ctl = wf_glob(sp.ctl);
    sp.hflag = wf_glob(sp.hflag);
    sp.U = wf_glob(sp.U);
    sp.pl_fx = wf_glob(sp.pl_fx);
    sp.pl_ix = wf_glob(sp.pl_ix);
    sp.pl_fy = wf_glob(sp.pl_fy);
    sp.pl_iy = wf_glob(sp.pl_iy);
    sp.pl_l = wf_glob(sp.pl_l);
    sp.pl_ru = wf_glob(sp.pl_ru);
    wf_glob_state(it.ys);
    wf_glob_state(it.yn);
    it.p = wf_glob(it.p);
    it.rho = wf_glob(it.rho);
    return it;
}

/* Complex value in the arithmetic type TA of a tridiagonal solve. */
template <typename TA>
struct alignas(2 * sizeof(TA)) wf_cx {
    TA x, y;
};
/* Entry i of a coefficient table in TA: the FP64 copy for TA = double. */
template <typename TA>
__device__ __forceinline__ TA wf_tab(const wf_real *t, const double *td, int i) {
    if constexpr (sizeof(TA) == sizeof(double))
        return td[i];
    else
        return (TA)t[i];
}

/* Thomas pivots of every (kx, ky) system (src/cu/pressure.cu:429-433):
 * u_0 = b_0, u_k = b_k - (a_{k-1}/u_{k-1}) c_{k-1}.  They do not change between
 * steps; the pivot entering each z-chunk of the tridiagonal solve (u_{k0-1},
 * k0 = chunk * lc) is stored once (FP64), and the solve re-forms the others
 * with the same operations in its own arithmetic type TA. */
template <typename TA>
__device__ __forceinline__ TA wf_pivot_next(const WfSpectral &sp, TA u, int k, TA K2, TA c0, TA *l_out) {
    const int nz = sp.nz;
    const TA ck1 = (k == 1) ? c0 : wf_tab<TA>(sp.tc, sp.tcd, k - 1);
    const TA bk = (k == nz - 1) ? -(K2 + (TA)sp.beta_top) : -(K2 + wf_tab<TA>(sp.beta, sp.betad, k));
    const TA l = wf_tab<TA>(sp.ta, sp.tad, k - 1) / u;
    *l_out = l;
    return bk - l * ck1;
}

/* The periodic copies on the top plane (whose unique nodes the solve never
 * writes), with the running max |p_new - p_old|, by one workgroup. */
__device__ __forceinline__ void wf_top_duplicates(const WfConst &c, wf_real *p, double &dmax) {
    const int kt = c.Nz - 1;
    for (int t = threadIdx.x; t < c.Ny + c.Nx - 1; t += blockDim.x) {
        long qd, qs;
        if (t < c.Ny) { /* i = Nx-1 from i = 0 */
            qd = wf_q(c, c.Nx - 1, t, kt);
            qs = wf_q(c, 0, (t == c.Ny - 1) ? 0 : t, kt);
        } else { /* j = Ny-1 from j = 0 */
            qd = wf_q(c, t - c.Ny, c.Ny - 1, kt);
            qs = wf_q(c, t - c.Ny, 0, kt);
        }
        wf_real v = p[qs];
        double d = (double)fabs(v - p[qd]);
        dmax = (d > dmax) ? d : dmax;
        p[qd] = v;
    }
}

}  // namespace WF_NS

#endif
